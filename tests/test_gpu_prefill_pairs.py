"""Prefill with two pairs of waves per row (launches of few rows): odd and even counts of active
blocks, rows with one block or none, ragged ends, and both sides of the rule that chooses it."""
from __future__ import annotations

import pytest
import torch

import attn_inputs as ai
from helpers import assert_close_bf16, require_gpu, to_np
from oracle import tasft_oracle as orc
from tasft_amd.kernels import BlockSparseFlashAttention

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["unit", "peaky"])
@pytest.mark.parametrize(("S", "Hq", "Hkv", "D", "bs", "causal"), [
    (448, 4, 2, 128, 64, True),      # 7 blocks: one pair
    (449, 4, 2, 128, 64, False),     # 8 blocks, one key in the last
    (1024, 32, 8, 128, 64, True),    # 512 rows
    (1025, 32, 8, 128, 64, True),    # 544 rows: one pair
    (2048, 32, 8, 64, 64, True),     # 1024 rows
    (2049, 32, 8, 64, 64, True),     # 1056 rows: one pair
    (1000, 32, 8, 64, 64, True),
    (4500, 2, 1, 128, 64, True),     # more than 64 key blocks per row
    (4200, 3, 3, 64, 128, False),
])
def test_few_rows(S, Hq, Hkv, D, bs, causal, kind):
    dev = require_gpu()
    nb = -(-S // bs)
    print(f"prefill pairs S={S} Hq={Hq} D={D} block {bs} causal={causal} {kind}", flush=True)
    q, k, v = ai.qkv(kind, (1, Hq, S, D), (1, Hkv, S, D), 21 + S, bs)
    mask = torch.rand(1, Hq, nb, nb, generator=torch.Generator().manual_seed(S)) < 0.3
    mask[:, 0] = torch.eye(nb, dtype=torch.bool)
    mask[:, 1, nb // 2] = False
    mask[:, -1, -2:] = True
    out = BlockSparseFlashAttention(block_size=bs, min_sparsity_for_speedup=0.0).forward(
        q.to(dev), k.to(dev), v.to(dev), mask.to(dev), causal=causal)
    torch.cuda.synchronize()
    ref = orc.attention_block_gather(to_np(q), to_np(k), to_np(v), mask.numpy(), bs, causal)
    assert_close_bf16(out, ref, f"prefill pairs S={S} D={D} block {bs} {kind}")
