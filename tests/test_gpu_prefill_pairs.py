"""Prefill with two pairs of waves per row (launches of few rows): odd and even counts of active
blocks, rows with one block or none, ragged ends, and both sides of the rule that chooses it."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import attn_inputs as ai
from helpers import MAX_ABS_TOL, assert_close_bf16, bar, require_gpu, to_np
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
    _check(S, Hq, Hkv, D, bs, causal, kind)


@pytest.mark.parametrize("kind", ["unit", "peaky"])
@pytest.mark.parametrize(("S", "Hq", "Hkv", "D", "bs", "causal"), [
    (4200, 8, 2, 128, 64, False),    # 528 rows
    (4200, 8, 2, 128, 128, True),    # 528 rows of 64 tokens
    (4200, 16, 4, 64, 64, False),    # 1056 rows
    (4200, 16, 4, 64, 128, True),
])
def test_one_pair_long_rows(S, Hq, Hkv, D, bs, causal, kind):
    """One pair, more than 64 key blocks per row and a ragged end. A row that attends to one key
    returns its V row, and among millions of values some exceed 4, where half a unit of the
    bf16 output is 2^-6 alone; P's rounding adds at most 2^-9 max|v|."""
    _check(S, Hq, Hkv, D, bs, causal, kind, rounding_bound=True)


def _check(S, Hq, Hkv, D, bs, causal, kind, rounding_bound=False):
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
    bound = MAX_ABS_TOL
    if rounding_bound:
        bound = max(bound, 2.0 ** (np.floor(np.log2(np.abs(ref).max())) - 8) + 2.0 ** -9 * float(v.abs().max()))
    assert_close_bf16(out, ref, f"prefill pairs S={S} D={D} block {bs} {kind}", max_abs=bound)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("causal", [True, False])
def test_packed_one_pair(causal, D):
    """A packed call above the row limits (the longest sequence's rows count for each), its
    first sequence of more than 64 key blocks."""
    dev = require_gpu()
    lens, Hq, Hkv = [4200, 700, 65], 8, 2
    cu = np.cumsum([0] + lens).tolist()
    print(f"prefill one pair packed D={D} causal={causal}", flush=True)
    nb = -(-max(lens) // 64)
    q, k, v = (t[0].transpose(0, 1).contiguous() for t in ai.qkv("unit", (1, Hq, cu[-1], D), (1, Hkv, cu[-1], D),
                                                                 7 + D, 64))
    mask = torch.rand(len(lens), Hq, nb, nb, generator=torch.Generator().manual_seed(D)) < 0.2
    mask |= torch.eye(nb, dtype=torch.bool)
    out = BlockSparseFlashAttention(block_size=64, min_sparsity_for_speedup=0.0).forward_varlen(
        q.to(dev), k.to(dev), v.to(dev), mask.to(dev), torch.tensor(cu, dtype=torch.int32), causal=causal)
    torch.cuda.synchronize()
    ref = orc.attention_varlen(to_np(q), to_np(k), to_np(v), cu, mask.numpy(), 64, causal)
    assert_close_bf16(out, ref, f"prefill one pair packed D={D} causal={causal}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(("S", "D"), [(440, 128), (512, 128), (440, 64), (512, 64)])  # one pair, two pairs
def test_nan_pattern(S, D, dtype):
    """A NaN in Q, K or V reaches the same outputs as in the oracle, whichever pair meets it."""
    dev = require_gpu()
    Hq, Hkv, nb = 4, 2, -(-S // 64)
    print(f"prefill pairs NaN S={S} D={D} {dtype}", flush=True)
    q, k, v = (t.float().to(dtype) for t in ai.qkv("unit", (1, Hq, S, D), (1, Hkv, S, D), 31 + S + D, 64))
    q[0, 0, 300, 5] = float("nan")
    k[0, 1, 130, 1] = float("nan")
    v[0, 0, 70, D - 1] = float("nan")
    mask = torch.rand(1, Hq, nb, nb, generator=torch.Generator().manual_seed(S)) < 0.5
    ref = orc.attention_block_gather(to_np(q), to_np(k), to_np(v), mask.numpy(), 64, True)
    assert np.isnan(ref).any() and not np.isnan(ref).all()
    out = BlockSparseFlashAttention(block_size=64, min_sparsity_for_speedup=0.0).forward(
        q.to(dev), k.to(dev), v.to(dev), mask.to(dev), causal=True)
    torch.cuda.synchronize()
    got, clean = to_np(out), ~np.isnan(ref)
    np.testing.assert_array_equal(np.isnan(got), ~clean)
    assert_close_bf16(np.where(clean, got, 0.0), np.where(clean, ref, 0.0), f"NaN S={S} D={D}", **bar(dtype))
