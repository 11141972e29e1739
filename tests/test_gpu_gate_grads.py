"""tasft_gate_grads (the gate's parameter gradients) at the edges of its tiles: row chunks of
16 to 64 query blocks, 16-key rounds, 64-unit tiles, 64-dim output tiles, the ends of the row
runs of the weight products (at most 128 rows each), and the block-diagonal cases, against the formula in 64 bits."""
from __future__ import annotations

import pytest
import torch

from helpers import require_gpu
from tasft_amd.modules import AttnGate
from tasft_amd.modules.attn_gate import _launch_gate

pytestmark = pytest.mark.gpu

CASES = [
    # B, Hq, Hkv, S, D, bs, hidden, causal
    (1, 1, 1, 40, 64, 64, 32, True),        # one query block, one key block
    (1, 2, 1, 1025, 64, 64, 1, True),       # 17 blocks (16-row chunks, two key rounds), one unit
    (2, 4, 4, 2048, 72, 32, 65, False),     # 64 blocks, a second unit tile of one unit, 72 dims
    (1, 8, 2, 16 * 65, 128, 16, 96, True),  # 65 blocks: a last chunk of one row
    (4, 32, 8, 32 * 66, 256, 32, 64, True), # 66 blocks in 64-row chunks, 256 dims, 2112 K rows
    (3, 6, 2, 700, 8, 64, 130, False),      # eight dims, a third unit tile of two units
    (8, 32, 8, 16 * 128, 128, 16, 72, True),  # 32768 rows, four tiles: the longest run, 128 rows
]


@pytest.mark.parametrize(("B", "Hq", "Hkv", "S", "D", "bs", "hidden", "causal"), CASES)
def test_parameter_gradients(B, Hq, Hkv, S, D, bs, hidden, causal):
    dev = require_gpu()
    print(f"gate grads B={B} Hq={Hq} Hkv={Hkv} S={S} D={D} bs={bs} hid={hidden} causal={causal}", flush=True)
    torch.manual_seed(S + hidden)
    gate = AttnGate(num_heads=Hq, head_dim=D, block_size=bs, gate_hidden_dim=hidden, is_causal=causal).to(dev)
    with torch.no_grad():
        gate.gate_proj_out.weight.mul_(30)
        gate.gate_proj_in.bias.normal_(std=0.05)
    g = torch.Generator(device=dev).manual_seed(S)
    q = torch.randn((B, Hq, S, D), generator=g, device=dev).to(torch.bfloat16)
    k = torch.randn((B, Hkv, S, D), generator=g, device=dev).to(torch.bfloat16)
    out = gate(q, k)
    r = torch.randn(out.soft_scores.shape, generator=g, device=dev)
    (out.soft_scores * r).sum().backward()
    got = {n: p.grad.double() for n, p in gate.named_parameters()}

    # The same sums in 64 bits from the forward's own units, block means and scores, so that
    # both sides agree on which units are active.
    fwd = _launch_gate(gate, q, k, gate._thresholds(0.5, dev), False, False, keep=True)
    nb = fwd["nb"]
    n_q = B * Hq * nb * hidden
    units = fwd["workspace"][: (n_q + B * Hkv * nb * hidden) * 4].view(torch.float32).double()
    u = units[:n_q].view(B, Hq, nb, hidden)
    v = units[n_q:].view(B, Hkv, nb, hidden).repeat_interleave(Hq // Hkv, 1)
    s = out.soft_scores.detach().double()
    grad = r.double() * s * (1 - s)
    w_out = gate.gate_proj_out.weight.detach().double().view(-1)
    du, dv = torch.empty_like(u), torch.empty_like(v)
    dw_out = torch.zeros(hidden, dtype=torch.float64, device=dev)
    for b in range(B):
        pre = u[b].unsqueeze(2) + v[b].unsqueeze(1)
        on = (pre > 0) * grad[b].unsqueeze(-1)
        du[b], dv[b] = on.sum(2) * w_out, on.sum(1) * w_out
        dw_out += (on * pre).sum((0, 1, 2))
    km = fwd["k_means"].double().repeat_interleave(Hq // Hkv, 1).reshape(-1, D)
    du, dv = du.reshape(-1, hidden), dv.reshape(-1, hidden)
    ref = {"gate_proj_in.weight": torch.cat([du.t() @ fwd["q_means"].double().reshape(-1, D), dv.t() @ km], 1),
           "gate_proj_in.bias": du.sum(0), "gate_proj_out.weight": dw_out.view(1, -1)}
    # fp32 sums in runs of at most 128 addends (2^-24 each) below 64-bit or pairwise ones: 128
    # roundings at most, and cancellation between addends of both signs; 1e-5 of the norm.
    for name, p in ref.items():
        err = float((got[name] - p).norm() / p.norm())
        assert err < 1e-5, f"{name}: {err:.2e}"
