"""C entries no Python path calls: the gate backward's partial sums per tile (tasft_gate_bwd)
against the reduced gradients of tasft_gate_grads, and the KL loss's partials without the sum
(tasft_gate_kl_fwd) against tasft_gate_kl_loss."""
from __future__ import annotations

import pytest
import torch

from helpers import require_gpu
from tasft_amd import _native
from tasft_amd.modules import AttnGate
from tasft_amd.modules.attn_gate import _launch_gate

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(("B", "Hq", "Hkv", "S", "D", "bs", "hidden", "causal"), [
    (1, 2, 1, 40, 64, 64, 32, True),        # one block
    (2, 4, 2, 32 * 33, 64, 32, 70, True),   # 33 blocks: a second tile of one, a second unit stage
    (1, 3, 3, 1000, 128, 16, 64, False),    # 63 blocks, non-causal
])
def test_gate_bwd_partials_add_up_to_the_gradients(B, Hq, Hkv, S, D, bs, hidden, causal):
    dev = require_gpu()
    print(f"gate_bwd B={B} Hq={Hq} S={S} bs={bs} hidden={hidden} causal={causal}", flush=True)
    torch.manual_seed(S)
    gate = AttnGate(num_heads=Hq, head_dim=D, block_size=bs, gate_hidden_dim=hidden, is_causal=causal).to(dev)
    with torch.no_grad():
        gate.gate_proj_out.weight.mul_(30)
    q = torch.randn(B, Hq, S, D, device=dev).bfloat16()
    k = torch.randn(B, Hkv, S, D, device=dev).bfloat16()
    f = _launch_gate(gate, q, k, gate._thresholds(0.5, dev), False, False, keep=True)
    soft, ws, nb = f["soft"], f["workspace"], f["nb"]
    gs = torch.randn_like(soft)
    w_out = gate.gate_proj_out.weight.detach().view(-1)
    lib, stream, flags = _native.load_library(), _native.stream_handle(dev), int(causal)

    n = lib.tasft_gate_bwd_workspace_bytes(B, Hq, S, bs, hidden)
    part = torch.full((n // 4,), float("nan"), device=dev)
    _native.check(lib.tasft_gate_bwd(soft.data_ptr(), gs.data_ptr(), ws.data_ptr(), ws.numel(), part.data_ptr(),
                                     n, B, Hq, Hkv, S, bs, hidden, flags, stream), "tasft_gate_bwd")
    tiles, plane = -(-nb // 32), B * Hq * nb * hidden
    part = part.double()
    got = {"du": part[: tiles * plane].view(tiles, B, Hq, nb, hidden).sum(0) * w_out,
           "dv": part[tiles * plane: 2 * tiles * plane].view(tiles, B, Hkv, Hq // Hkv, nb, hidden).sum((0, 3)) * w_out,
           "dw_out": part[2 * tiles * plane:].view(-1, hidden).sum(0)}

    ref = {"du": torch.empty(B, Hq, nb, hidden, device=dev), "dv": torch.empty(B, Hkv, nb, hidden, device=dev),
           "dw_out": torch.empty(hidden, device=dev)}
    dw, db = torch.empty(hidden, 2 * D, device=dev), torch.empty(hidden, device=dev)
    n = lib.tasft_gate_grads_workspace_bytes(B, Hq, Hkv, S, D, bs, hidden)
    tmp = torch.empty(n, dtype=torch.uint8, device=dev)
    _native.check(lib.tasft_gate_grads(
        soft.data_ptr(), gs.data_ptr(), ws.data_ptr(), ws.numel(), f["q_means"].data_ptr(), f["k_means"].data_ptr(),
        w_out.data_ptr(), ref["du"].data_ptr(), ref["dv"].data_ptr(), dw.data_ptr(), db.data_ptr(),
        ref["dw_out"].data_ptr(), tmp.data_ptr(), n, B, Hq, Hkv, S, D, bs, hidden, flags, stream), "tasft_gate_grads")
    for name, r in ref.items():
        # Two orders of the same fp32 sums, runs of at most 64 addends of both signs.
        assert float((got[name] - r.double()).norm() / r.double().norm()) < 1e-5, name


@pytest.mark.parametrize("n", [37, 128, 160])  # scores in registers up to 128 x 128, streamed above
def test_kl_fwd_is_kl_loss_without_the_sum(n):
    dev = require_gpu()
    B, H = 2, 3
    print(f"kl_fwd {n} x {n}", flush=True)
    g = torch.Generator(device=dev).manual_seed(n)
    soft = torch.rand(B, H, n, n, generator=g, device=dev).tril()
    target = torch.rand(B, H, n, n, generator=g, device=dev).tril()
    target /= target.sum((2, 3), keepdim=True)
    lib, stream = _native.load_library(), _native.stream_handle(dev)
    part, part2 = torch.empty(B * H, device=dev), torch.empty(B * H, device=dev)
    grad, grad2, loss = torch.empty_like(soft), torch.empty_like(soft), torch.empty((), device=dev)
    status = torch.zeros(3, dtype=torch.int32, device=dev)
    args = (soft.data_ptr(), target.data_ptr(), B, H, n, n)
    _native.check(lib.tasft_gate_kl_fwd(*args, part.data_ptr(), grad.data_ptr(), stream), "tasft_gate_kl_fwd")
    _native.check(lib.tasft_gate_kl_loss(*args, part2.data_ptr(), grad2.data_ptr(), loss.data_ptr(),
                                         status.data_ptr(), stream), "tasft_gate_kl_loss")
    assert torch.equal(part, part2) and torch.equal(grad, grad2) and status.tolist()[:2] == [0, 0]
    assert float(loss) == pytest.approx(float(part.double().sum() / B), rel=1e-7)
    _native.check(lib.tasft_gate_kl_fwd(*args, part.data_ptr(), None, stream), "tasft_gate_kl_fwd")
    assert torch.equal(part, part2)
    u = soft.double() / (soft.double().sum((2, 3), keepdim=True) + 1e-8) + 1e-8
    t = target.double()
    ref = torch.where(t > 0, t * (t.clamp_min(1e-300).log() - u.log()), 0.0).sum((2, 3)).view(-1)
    # Each grid's sum of t = 1 weighs logarithms of order 10 that round by 2^-24.
    torch.testing.assert_close(part.double(), ref, rtol=0, atol=1e-5)
