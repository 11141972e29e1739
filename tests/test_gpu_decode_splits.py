"""Decode at the edges of its selection pass and of the merge of splits: rows of 255 to 257 key
blocks (one pass over the mask, or two), 1 to 16 query heads per KV head (mask bytes are read
eight heads at a time), and split counts around the merge's four shares of eight."""
from __future__ import annotations

import pytest
import torch

from helpers import assert_close_bf16, require_gpu, to_np
from oracle import tasft_oracle as orc
from tasft_amd import workloads as wl
from tasft_amd.kernels import BlockSparseFlashAttention

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(("G", "nb", "splits"), [
    (1, 3, 2), (7, 256, 3), (8, 255, 4), (9, 257, 5), (16, 256, 31), (4, 257, 32), (3, 70, 33),
    (2, 256, 100), (5, 257, 257),
])
def test_decode_selection_and_merge(G, nb, splits):
    dev = require_gpu()
    B, Hkv, D, bs = 2, 2, 64, 32
    S = nb * bs - 5
    print(f"decode G={G} blocks={nb} splits={splits}", flush=True)
    q = wl.randn_bf16((B, G * Hkv, 1, D), 31, scale=1.0)
    k = wl.randn_bf16((B, Hkv, S, D), 32, scale=1.0)
    v = wl.randn_bf16((B, Hkv, S, D), 33, scale=1.0)
    mask = torch.rand((B, G * Hkv, 1, nb), generator=torch.Generator().manual_seed(G * nb)) < 0.3
    mask[1, 0] = False  # a head without a block
    mask[:, -1, 0, -1] = True
    bsfa = BlockSparseFlashAttention(block_size=bs, min_sparsity_for_speedup=0.0)
    dv = [t.to(dev) for t in (q, k, v, mask)]
    out = bsfa.forward_decode(*dv, num_splits=splits)
    ref = orc.sparse_decode(to_np(q), to_np(k), to_np(v), mask.numpy(), bs)
    assert_close_bf16(out, ref, f"decode G={G} blocks={nb} splits={splits}")
    assert not out[1, 0].any()
