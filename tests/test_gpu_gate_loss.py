"""``gate_loss_from_qk``'s checks and its fused sum: NaN and infinities in the scores and in the
mask, scores in 16 and 64 bits, and the loss of one and of many (batch, head) grids."""
from __future__ import annotations

import pytest
import torch

from helpers import require_gpu
from tasft_amd import workloads as wl
from tasft_amd.exceptions import KernelError, NaNDetectedError
from tasft_amd.training import TASFTObjective, gate_loss_from_qk, gate_target_from_qk

pytestmark = pytest.mark.gpu


def _inputs(B, Hq, Hkv, S, bs, dev):
    q, k, _ = (t.to(dev) for t in wl.qkv(wl.Shape(B, Hq, Hkv, S, 64), 17))
    nb = -(-S // bs)
    g = torch.Generator().manual_seed(S)
    soft = torch.sigmoid(torch.randn(B, Hq, nb, nb, generator=g)).tril().to(dev)
    return q, k, soft


@pytest.mark.parametrize(("B", "Hq", "Hkv", "S", "bs"), [
    (1, 1, 1, 60, 64),       # one value in one grid
    (3, 64, 8, 200, 64),     # 192 grids: the last workgroup adds the parts
    (2, 600, 600, 70, 32),   # more grids than the workgroup has threads
    (1, 2, 1, 4200, 32),     # 132 x 132 blocks: the streaming kernel
])
def test_loss_is_the_reference_sum(B, Hq, Hkv, S, bs):
    dev = require_gpu()
    print(f"gate loss B={B} Hq={Hq} S={S} bs={bs}", flush=True)
    q, k, soft = _inputs(B, Hq, Hkv, S, bs, dev)
    target = gate_target_from_qk(q, k, bs)
    ref = TASFTObjective.compute_gate_loss(soft.double(), target.double())
    for dtype in (torch.float32, torch.float64):
        s = soft.clone().to(dtype).requires_grad_(True)
        loss = gate_loss_from_qk(s, q, k, bs)
        loss.backward()
        # A 64-bit sum of fp32 grids, each a sum of at most 17424 terms of both signs; the two
        # logarithms of a term round by 2^-24 of values of order 10, weighted by sum t = 1 a grid.
        assert float(loss.detach()) == pytest.approx(float(ref), rel=1e-5, abs=2e-6 * Hq)
        assert s.grad.dtype == dtype


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float64])
@pytest.mark.parametrize(("value", "nan", "inf"), [(float("nan"), True, False), (float("inf"), False, True),
                                                   (-float("inf"), False, True)])
def test_non_finite_scores_are_rejected(value, nan, inf, dtype):
    dev = require_gpu()
    q, k, soft = _inputs(2, 4, 2, 300, 64, dev)
    soft = soft.to(dtype)
    gate_loss_from_qk(soft, q, k, 64)
    soft[1, 3, 4, 2] = value
    with pytest.raises(NaNDetectedError, match=f"gate_soft_scores: NaN={nan}, Inf={inf}") as e:
        gate_loss_from_qk(soft, q, k, 64)
    assert e.value.context["dtype"] == str(dtype) and e.value.context["shape"] == [2, 4, 5, 5]


@pytest.mark.parametrize("form", ["row", "full", "expanded", "int"])
def test_mask_is_checked_and_padded(form):
    """-inf and the lowest value pass, NaN and +inf are rejected (before the scores), and a
    transposed or expanded mask reads as its contiguous copy."""
    dev = require_gpu()
    S = 131
    q, k, soft = _inputs(2, 4, 2, S, 64, dev)
    lowest = torch.finfo(torch.float32).min
    if form == "row":
        mask = torch.zeros(2, S, device=dev)
        mask[1, 70:] = lowest
    elif form == "int":
        mask = torch.randint(0, 3, (2, S), device=dev)
    else:
        mask = torch.randn(2, 1, S, S, device=dev).transpose(2, 3)
        mask[0, 0, 5, 3] = -float("inf")
        if form == "expanded":
            mask = mask[:1, :, :, :].expand(2, 4, S, S)
    a = gate_target_from_qk(q, k, 64, attention_mask=mask)
    b = gate_target_from_qk(q, k, 64, attention_mask=mask.clone(memory_format=torch.contiguous_format))
    assert torch.equal(a, b)
    if form == "int":
        return
    for value, nan, inf in ((float("nan"), True, False), (float("inf"), False, True)):
        bad = mask.clone(memory_format=torch.contiguous_format)
        bad.view(-1)[-1] = value
        soft[0, 0, 0, 0] = float("nan")
        for call in (lambda: gate_target_from_qk(q, k, 64, attention_mask=bad),
                     lambda: gate_loss_from_qk(soft, q, k, 64, attention_mask=bad)):
            with pytest.raises(NaNDetectedError, match=f"attn_scores: NaN={nan}, Inf={inf}"):
                call()
    with pytest.raises(KernelError, match="do not match"):
        gate_loss_from_qk(soft[:, :, :2], q, k, 64, attention_mask=mask)
