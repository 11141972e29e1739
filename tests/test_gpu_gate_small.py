"""The gate around the line between its two forms at block 64 (up to 256 chunks of 16 blocks: a
pooling launch of four blocks per workgroup and the pairwise tiles; above: one kernel): ends of
a four-block group, both head dims, and the two forms' agreement on the same heads."""
from __future__ import annotations

import pytest
import torch

from helpers import require_gpu
from tasft_amd.modules import AttnGate

pytestmark = pytest.mark.gpu


def _gate(Hq, D, hidden, causal, dev):
    torch.manual_seed(hidden)
    gate = AttnGate(num_heads=Hq, head_dim=D, block_size=64, gate_hidden_dim=hidden, is_causal=causal)
    with torch.no_grad():
        gate.gate_proj_out.weight.mul_(20)
        gate.gate_proj_in.bias.normal_(std=0.1)
    return gate.to(dev).requires_grad_(False)


def _exact(gate, q, k):
    D = q.shape[-1]
    w = gate.gate_proj_in.weight.double()
    u = gate._pool_to_blocks(q.double()) @ w[:, :D].t() + gate.gate_proj_in.bias.double()
    v = gate._pool_to_blocks(k.double()) @ w[:, D:].t()
    v = v.repeat_interleave(q.shape[1] // k.shape[1], 1)
    logits = torch.relu(u.unsqueeze(3) + v.unsqueeze(2)) @ gate.gate_proj_out.weight.double().view(-1)
    soft = torch.sigmoid(logits)
    return soft.tril() if gate.is_causal else soft


@pytest.mark.parametrize(("B", "Hq", "Hkv", "S", "D", "hidden", "causal", "dtype"), [
    (1, 1, 1, 1, 128, 32, True, torch.bfloat16),        # one token
    (2, 4, 2, 64 * 4, 64, 48, False, torch.float16),    # exactly one group; hidden not of 32
    (1, 8, 2, 64 * 5 + 1, 128, 128, True, torch.bfloat16),
    (4, 32, 32, 900, 64, 32, True, torch.bfloat16),     # 256 chunks: the last small launch
    (4, 33, 33, 900, 64, 32, True, torch.bfloat16),     # 264 chunks: one kernel
    (2, 16, 2, 9000, 128, 32, True, torch.bfloat16),    # one kernel: 141 blocks, two key groups
    (8, 24, 8, 1300, 64, 64, False, torch.float16),     # one kernel, non-causal, partial chunk
    (8, 28, 4, 1000, 128, 96, True, torch.bfloat16),    # one kernel, ragged last block
])
def test_both_forms(B, Hq, Hkv, S, D, hidden, causal, dtype):
    dev = require_gpu()
    print(f"gate B={B} Hq={Hq} Hkv={Hkv} S={S} D={D} hidden={hidden} causal={causal}", flush=True)
    gate = _gate(Hq, D, hidden, causal, dev)
    g = torch.Generator(device=dev).manual_seed(S)
    q = torch.randn(B, Hq, S, D, generator=g, device=dev).to(dtype)
    k = torch.randn(B, Hkv, S, D, generator=g, device=dev).to(dtype)
    out = gate(q, k, threshold=0.5, force_diagonal=True)
    ref = _exact(gate, q, k)
    # fp32 sums of 64 + D + hidden terms, a sigmoid.
    torch.testing.assert_close(out.soft_scores.double(), ref, rtol=0, atol=2e-6)
    on = (out.soft_scores >= 0.5) | torch.eye(ref.shape[-1], dtype=torch.bool, device=dev)
    assert torch.equal(out.hard_mask, on)
    assert out.sparsity_ratio == pytest.approx(1 - on.double().mean().item(), abs=1e-9)


def test_forms_agree_on_the_same_heads():
    """A batch above the limit (one kernel) against its entries alone (two launches)."""
    dev = require_gpu()
    B, Hq, Hkv, S, D, hidden = 8, 28, 4, 1100, 128, 64  # 512 chunks; 64 each
    gate = _gate(Hq, D, hidden, True, dev)
    g = torch.Generator(device=dev).manual_seed(S)
    q = torch.randn(B, Hq, S, D, generator=g, device=dev).bfloat16()
    k = torch.randn(B, Hkv, S, D, generator=g, device=dev).bfloat16()
    both = gate(q, k, threshold=0.5)
    for b in range(B):
        one = gate(q[b:b + 1], k[b:b + 1], threshold=0.5)
        # Two orders of the fp32 sums, each within 2e-6 of the exact score (test_both_forms).
        torch.testing.assert_close(one.soft_scores, both.soft_scores[b:b + 1], rtol=0, atol=4e-6)
