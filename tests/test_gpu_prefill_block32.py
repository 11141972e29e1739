"""The block-32 prefill kernel (one wave per 32 query rows, tiles gathered from one or two
active blocks) where it can go wrong: every count of active blocks a row can have at its
start, a last block of one to 32 rows, rows of more than one mask word, and token strides the
32-bit offsets do not cover."""
from __future__ import annotations

import pytest
import torch

from helpers import assert_close_bf16, require_gpu, to_np
from oracle import tasft_oracle as orc
from tasft_amd import workloads as wl
from tasft_amd.kernels import BlockSparseFlashAttention

pytestmark = pytest.mark.gpu


def _attn(q, k, v, mask, causal=True):
    out = BlockSparseFlashAttention(block_size=32, min_sparsity_for_speedup=0.0).forward(
        q, k, v, mask, causal=causal)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize(("S", "causal"), [(1, True), (32, True), (33, False), (161, True), (223, False),
                                           (2200, True)])
def test_counts_of_active_blocks(S, causal, D):
    """Query block i of head h attends to (i + h) % 4 blocks, spread over the row: empty
    rows, and odd and even counts (a gathered tile with and without its second block)."""
    dev = require_gpu()
    B, Hq, Hkv = 2, 4, 2
    nb = -(-S // 32)
    print(f"block 32 S={S} D={D} causal={causal}", flush=True)
    mask = torch.zeros(B, Hq, nb, nb, dtype=torch.bool)
    for h in range(Hq):
        for i in range(nb):
            reach = i + 1 if causal else nb
            for c in range((i + h) % 4):
                mask[:, h, i, reach - 1 - (c * reach) // 3] = True
    q = wl.randn_bf16((B, Hq, S, D), 71, scale=1.0)
    k = wl.randn_bf16((B, Hkv, S, D), 72, scale=1.0)
    v = wl.randn_bf16((B, Hkv, S, D), 73, scale=1.0)
    out = _attn(q.to(dev), k.to(dev), v.to(dev), mask.to(dev), causal)
    ref = orc.attention_block_gather(to_np(q), to_np(k), to_np(v), mask.numpy(), 32, causal)
    assert_close_bf16(out, ref, f"block 32 S={S} D={D}")
    empty = torch.arange(S) // 32 % 4 == 0  # head 0: (i + 0) % 4 == 0
    assert not out[:, 0, empty.to(dev)].any()


@pytest.mark.parametrize("wide", ["k", "v", "q"])
def test_token_stride_beyond_32_bit_offsets(wide):
    """One tensor's rows 2 GB and more apart in all (the 64-bit address path), equal to the
    contiguous call bit for bit; K repeated by a zero token stride as well."""
    dev = require_gpu()
    S, D, pitch = 75, 64, 1 << 24
    t = {n: wl.randn_bf16((1, 2, S, D), 80 + i, scale=1.0).to(dev) for i, n in enumerate("qkv")}
    mask = (torch.rand(1, 2, 3, 3, generator=torch.Generator().manual_seed(9)) < 0.7).to(dev)
    ref = _attn(t["q"], t["k"], t["v"], mask, causal=False)
    buf = torch.empty(S * pitch, dtype=torch.bfloat16, device=dev)
    view = buf.as_strided((1, 2, S, D), (0, D, pitch, 1))
    view.copy_(t[wide])
    out = _attn(*(view if n == wide else t[n] for n in "qkv"), mask, causal=False)
    assert torch.equal(out, ref)
    same = t["k"][:, :, :1].expand(1, 2, S, D)
    assert torch.equal(_attn(t["q"], same, t["v"], mask), _attn(t["q"], same.contiguous(), t["v"], mask))
