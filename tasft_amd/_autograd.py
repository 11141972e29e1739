"""Autograd helper shared by the functions whose backward runs kernels."""
from __future__ import annotations

import functools

import torch
from torch.autograd.function import once_differentiable


def first_order_only(backward):
    """``once_differentiable``, entered only while a graph of the gradients is being built
    (``create_graph=True``): a second derivative is refused instead of formed from the torch
    operations around the kernels alone. Its wrapper takes 4.4 us of host time per call; in an
    ordinary backward there is no graph to cut."""
    once = once_differentiable(backward)

    @functools.wraps(backward)
    def run(ctx, *grads):
        return (once if torch.is_grad_enabled() else backward)(ctx, *grads)

    return run


__all__ = ["first_order_only"]
