"""tasft_gate_decode_rows_fwd at the edges of its thread layout: hidden widths of one and of
several 32-unit lanes' shares up to 256, head dims from 8 to 256 split over up to 32 threads,
one to eight heads per KV head, and rows around the 128 key blocks of a pass, against the
formula in 64 bits."""
from __future__ import annotations

import ctypes

import pytest
import torch

from helpers import require_gpu
from tasft_amd import _native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("reset", [0, 1])
@pytest.mark.parametrize(("B", "Hkv", "G", "D", "hid", "row"), [
    (1, 1, 1, 8, 4, 0),
    (2, 3, 2, 64, 36, 127),
    (1, 2, 7, 128, 32, 128),
    (3, 2, 4, 72, 128, 129),
    (1, 4, 8, 256, 256, 300),
    (2, 1, 3, 128, 132, 17),
])
def test_decode_rows(B, Hkv, G, D, hid, row, reset):
    dev = require_gpu()
    print(f"decode rows B={B} Hkv={Hkv} G={G} D={D} hidden={hid} row={row} reset={reset}", flush=True)
    Hq = Hkv * G
    g = torch.Generator(device=dev).manual_seed(D + hid + row)
    rnd = lambda *shape: torch.randn(*shape, generator=g, device=dev)  # noqa: E731
    q, k = rnd(B, Hq, D).bfloat16(), rnd(B, Hkv, D).bfloat16()
    qs, ks, uk = rnd(B, Hq, D), rnd(B, Hkv, D), rnd(B, Hkv, row + 3, hid)
    wq, wk, b_in, w_out = rnd(D, hid) / 16, rnd(D, hid) / 16, rnd(hid), rnd(hid) / 8
    tau = torch.rand(Hq, generator=g, device=dev)
    q_sum, k_sum, units = qs.clone(), ks.clone(), uk.clone()
    soft = torch.empty(B, Hq, row + 1, device=dev)
    mask = torch.empty(B, Hq, row + 1, dtype=torch.uint8, device=dev)
    count = torch.empty(1, dtype=torch.int64, device=dev)
    st = lambda t: (ctypes.c_int64 * 2)(*t.stride()[:2])  # noqa: E731
    lib = _native.load_library()
    rc = lib.tasft_gate_decode_rows_fwd(
        q.data_ptr(), k.data_ptr(), st(q), st(k), q_sum.data_ptr(), k_sum.data_ptr(), units.data_ptr(),
        units.stride(1), wq.data_ptr(), wk.data_ptr(), b_in.data_ptr(), w_out.data_ptr(), tau.data_ptr(),
        soft.data_ptr(), mask.data_ptr(), count.data_ptr(), B, Hq, Hkv, D, hid, row, reset, 3, 0,
        _native.stream_handle(dev))
    _native.check(rc, "tasft_gate_decode_rows_fwd")
    torch.cuda.synchronize()
    q2 = q.double() + (0 if reset else qs.double())
    k2 = k.double() + (0 if reset else ks.double())
    v = uk.double().clone()
    v[:, :, row] = k2 @ wk.double()
    u = q2 @ wq.double() + b_in.double()
    pre = u.unsqueeze(2) + v[:, :, : row + 1].repeat_interleave(G, 1)
    ref = torch.sigmoid(torch.relu(pre) @ w_out.double())
    # fp32 sums: (D + hidden) roundings of 2^-24 on logits of order 10 at most, and a sigmoid
    # (slope 1/4).
    torch.testing.assert_close(soft.double(), ref, rtol=0, atol=1e-5)
    torch.testing.assert_close(units.double()[:, :, row], v[:, :, row], rtol=0, atol=1e-4)
    assert torch.equal(units[:, :, :row], uk[:, :, :row]) and torch.equal(units[:, :, row + 1:], uk[:, :, row + 1:])
    torch.testing.assert_close(q_sum.double(), q2, rtol=1e-6, atol=1e-6)
    torch.testing.assert_close(k_sum.double(), k2, rtol=1e-6, atol=1e-6)
    on = soft >= tau.view(1, -1, 1)
    on[:, :, row] = True
    assert torch.equal(mask.bool(), on) and int(count) == int(on.sum())
