"""The two-wave prefill kernel at head dim 64: ends of tiles and rows, scores that make the exp2
reference move or stay within its margin, and token strides below D and beyond 32-bit offsets."""
from __future__ import annotations

import pytest
import torch

import attn_inputs as ai
from helpers import assert_close_bf16, require_gpu, to_np
from oracle import tasft_oracle as orc
from tasft_amd.kernels import BlockSparseFlashAttention

pytestmark = pytest.mark.gpu


def _attn(q, k, v, mask, bs, causal=True):
    out = BlockSparseFlashAttention(block_size=bs, min_sparsity_for_speedup=0.0).forward(
        q, k, v, mask, causal=causal)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("kind", ["unit", "peaky"])
@pytest.mark.parametrize(("S", "bs", "causal"), [(1, 64, True), (63, 64, False), (65, 64, True), (4200, 64, True),
                                                 (129, 128, False), (1000, 128, True)])
def test_ends_of_tiles(S, bs, causal, kind):
    dev = require_gpu()
    B, Hq, Hkv, D = 1, 4, 2, 64
    nb = -(-S // bs)
    print(f"prefill D=64 S={S} block {bs} causal={causal} {kind}", flush=True)
    q, k, v = ai.qkv(kind, (B, Hq, S, D), (B, Hkv, S, D), 11 + S, bs)
    mask = torch.rand(B, Hq, nb, nb, generator=torch.Generator().manual_seed(S)) < 0.4
    mask[:, 1, nb // 2] = False
    out = _attn(q.to(dev), k.to(dev), v.to(dev), mask.to(dev), bs, causal)
    ref = orc.attention_block_gather(to_np(q), to_np(k), to_np(v), mask.numpy(), bs, causal)
    assert_close_bf16(out, ref, f"prefill D=64 S={S} block {bs} {kind}")


def test_token_strides():
    """Q rows 2 GB and more apart in all, and rows repeated by a zero token stride, equal the
    contiguous call bit for bit."""
    dev = require_gpu()
    S, D, pitch = 140, 64, 1 << 23
    q, k, v = (t.to(dev) for t in ai.qkv("unit", (1, 2, S, D), (1, 2, S, D), 5, 64))
    mask = torch.ones(1, 2, 3, 3, dtype=torch.bool, device=dev)
    ref = _attn(q, k, v, mask, 64)
    buf = torch.empty(S * pitch, dtype=torch.bfloat16, device=dev)
    far = buf.as_strided((1, 2, S, D), (0, D, pitch, 1))
    far.copy_(q)
    assert torch.equal(_attn(far, k, v, mask, 64), ref)
    for i in range(3):
        t = [q, k, v]
        t[i] = t[i][:, :, :1].expand(1, 2, S, D)
        c = [x.contiguous() for x in t]
        assert torch.equal(_attn(*t, mask, 64), _attn(*c, mask, 64))
