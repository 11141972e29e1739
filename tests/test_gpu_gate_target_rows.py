"""The one-wave gate-target kernel's packing of (head, query block) rows four to a workgroup:
group sizes that leave waves on different query blocks or without a row, against the oracle,
and a key-padding row against the same mask given per query (another kernel), bit for bit."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import require_gpu, to_np
from oracle import tasft_oracle as orc
from tasft_amd import workloads as wl
from tasft_amd.training import gate_target_from_qk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize(("B", "Hq", "Hkv", "S", "D", "bs"), [
    (1, 1, 1, 50, 128, 64),     # one row: three waves without one
    (2, 3, 1, 333, 64, 64),     # G=3, six query blocks: 18 rows, a last workgroup of two
    (1, 7, 1, 450, 128, 32),    # G=7, 32-token output blocks
    (2, 8, 8, 300, 128, 128),   # G=1: four query blocks to a workgroup, pooled
    (1, 12, 2, 190, 64, 64),    # G=6
    (1, 4, 1, 1300, 64, 64),    # 21 blocks a row: runs of eight, the last of five
    (1, 3, 1, 1090, 128, 32),   # rows ending in different runs of one workgroup
    (2, 1, 1, 1160, 64, 128),   # runs of a pooled output
])
def test_rows_packed_four_to_a_workgroup(B, Hq, Hkv, S, D, bs, causal):
    dev = require_gpu()
    print(f"gate target rows B={B} Hq={Hq} Hkv={Hkv} S={S} D={D} bs={bs} causal={causal}", flush=True)
    q = wl.randn_bf16((B, Hq, S, D), 91, scale=1.0)
    k = wl.randn_bf16((B, Hkv, S, D), 92, scale=1.0)
    qd, kd = q.to(dev), k.to(dev)
    raw = to_np(gate_target_from_qk(qd, kd, bs, causal=causal, normalize="none"))
    ref = orc.block_max(to_np(q), to_np(k), bs, causal=causal)
    fin = np.isfinite(ref)
    assert (np.isfinite(raw) == fin).all()
    # fp32 sums of D exact products of 16-bit values, in another order: D roundings of 2^-24
    # of partial sums of order sqrt(D), scaled by 1/sqrt(D).
    np.testing.assert_allclose(raw[fin], ref[fin], rtol=0, atol=4e-5)

    mask = torch.randn(B, S, device=dev)
    mask[:, S // 2:] = torch.finfo(torch.float32).min
    mask[0, S // 3] = -float("inf")
    row = gate_target_from_qk(qd, kd, bs, causal=causal, normalize="none", attention_mask=mask)
    full = gate_target_from_qk(qd, kd, bs, causal=causal, normalize="none",
                               attention_mask=mask[:, None, None, :].expand(B, 1, S, S))
    assert torch.equal(row, full)
