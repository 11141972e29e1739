"""Second derivatives through the gate's and the KL loss's autograd functions are refused: their
backwards run kernels, so a graph of their results could only hold a part of the derivative.
The functions are the real ones, on the CPU, with kernel calls that do nothing."""
from __future__ import annotations

import pytest
import torch

from tasft_amd import _native
from tasft_amd.modules import AttnGate
from tasft_amd.modules.attn_gate import _HipGateFunction
from tasft_amd.training.objectives import _GateKL


class _NoKernels:
    def __getattr__(self, name):
        return (lambda *a: 256) if name.endswith("_bytes") else (lambda *a: 0)


@pytest.fixture(autouse=True)
def _stub(monkeypatch):
    monkeypatch.setattr(_native, "load_library", _NoKernels)
    monkeypatch.setattr(_native, "stream_handle", lambda device: 0)


@pytest.mark.parametrize("wrt", ["q", "k", "w"])
@pytest.mark.parametrize("power", [1, 2])  # the gradient of the scores: without and with a graph
def test_gate_refuses_a_second_backward(wrt, power):
    gate = AttnGate(num_heads=2, head_dim=64, gate_hidden_dim=32)
    q = torch.randn(1, 2, 128, 64).bfloat16().requires_grad_(True)
    k = torch.randn(1, 1, 128, 64).bfloat16().requires_grad_(True)
    soft, _, _ = _HipGateFunction.apply(q, k, gate.gate_proj_in.weight, gate.gate_proj_in.bias,
                                        gate.gate_proj_out.weight, gate, torch.full((2,), 0.5), False)
    x = {"q": q, "k": k, "w": gate.gate_proj_in.weight}[wrt]
    (g,) = torch.autograd.grad((soft ** power).sum(), x, create_graph=True)
    assert g.shape == x.shape
    with pytest.raises(RuntimeError, match="does not require grad|once_differentiable"):
        g.float().pow(2).sum().backward()


@pytest.mark.parametrize("power", [1, 2])
def test_loss_refuses_a_second_backward(power):
    soft = torch.rand(1, 2, 3, 3, requires_grad=True)
    loss = _GateKL.apply(soft, torch.rand(1, 2, 3, 3))
    (g,) = torch.autograd.grad(loss ** power, soft, create_graph=True)
    with pytest.raises(RuntimeError, match="does not require grad|once_differentiable"):
        g.sum().backward()
