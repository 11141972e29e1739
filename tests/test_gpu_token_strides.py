"""Token strides below the head dim (one row repeated by a stride of 0, rows that overlap): each
call equals the one on contiguous copies."""
from __future__ import annotations

import pytest
import torch

from helpers import require_gpu
from tasft_amd import workloads as wl
from tasft_amd.kernels import BlockSparseFlashAttention
from tasft_amd.modules import AttnGate
from tasft_amd.training import gate_target_from_qk

pytestmark = pytest.mark.gpu


def _views(heads, S, D, seed, dev):
    """[1, heads, S, D] of one row a head, and of rows eight elements apart."""
    row = wl.randn_bf16((1, heads, 1, D), seed, scale=1.0).to(dev).expand(1, heads, S, D)
    pool = wl.randn_bf16((heads, 8 * S + D), seed + 1, scale=1.0).to(dev)
    return row, pool.as_strided((1, heads, S, D), (0, pool.stride(0), 8, 1))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("bs", [32, 64, 128])
def test_prefill(bs, D):
    dev = require_gpu()
    S, Hq, Hkv = 333, 4, 2
    print(f"prefill token strides block {bs} D={D}", flush=True)
    q, k, v = (wl.randn_bf16((1, h, S, D), 5 + i, scale=1.0).to(dev) for i, h in enumerate((Hq, Hkv, Hkv)))
    nb = -(-S // bs)
    mask = (torch.rand(1, Hq, nb, nb, generator=torch.Generator().manual_seed(bs)) < 0.7).to(dev)
    mask |= torch.eye(nb, dtype=torch.bool, device=dev)
    attn = BlockSparseFlashAttention(block_size=bs, min_sparsity_for_speedup=0.0)
    cu = torch.tensor([0, S - 100, S], device=dev)
    varlen_mask = mask[..., :nb, :nb].expand(2, Hq, nb, nb)
    for i in range(3):
        for view in _views((Hq, Hkv, Hkv)[i], S, D, 20 + i, dev):
            t = [q, k, v]
            t[i] = view
            c = [x.contiguous() for x in t]
            assert torch.equal(attn.forward(*t, mask, causal=True), attn.forward(*c, mask, causal=True))
            t, c = ([x[0].transpose(0, 1) for x in y] for y in (t, c))
            assert torch.equal(attn.forward_varlen(*t, varlen_mask, cu, S),
                               attn.forward_varlen(*c, varlen_mask, cu, S))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize(("B", "bs"), [(1, 32), (1, 64), (8, 64), (1, 128)])  # 8: the one-launch form
def test_gate(B, bs, D):
    dev = require_gpu()
    S, Hq, Hkv = 1100, 32, 8
    print(f"gate token strides B={B} block {bs} D={D}", flush=True)
    torch.manual_seed(bs + D)
    gate = AttnGate(num_heads=Hq, head_dim=D, block_size=bs, gate_hidden_dim=32).to(dev).requires_grad_(False)
    q, k = (wl.randn_bf16((B, h, S, D), 41 + i, scale=1.0).to(dev) for i, h in enumerate((Hq, Hkv)))
    for i in range(2):
        for view in _views((Hq, Hkv)[i], S, D, 50 + i, dev):
            t = [q, k]
            t[i] = view.expand(B, -1, -1, -1)
            a = gate(*t, threshold=0.5)
            b = gate(*(x.contiguous() for x in t), threshold=0.5)
            # Another kernel pools such rows, with its fp32 sums in another order: bs + D + hidden
            # terms of 2^-24 on logits of order one, and a sigmoid (slope 1/4).
            torch.testing.assert_close(a.soft_scores, b.soft_scores, rtol=0, atol=2e-6)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("bs", [32, 64, 128])
def test_gate_target(bs, D):
    dev = require_gpu()
    S, Hq, Hkv = 333, 4, 2
    print(f"gate target token strides block {bs} D={D}", flush=True)
    q, k = (wl.randn_bf16((1, h, S, D), 61 + i, scale=1.0).to(dev) for i, h in enumerate((Hq, Hkv)))
    per_query = torch.randn(1, 1, S, S, device=dev)
    for i in range(2):
        for view in _views((Hq, Hkv)[i], S, D, 70 + i, dev):
            t = [q, k]
            t[i] = view
            c = [x.contiguous() for x in t]
            for mask in (None, per_query[:, 0, 0], per_query):
                assert torch.equal(gate_target_from_qk(*t, bs, normalize="none", attention_mask=mask),
                                   gate_target_from_qk(*c, bs, normalize="none", attention_mask=mask))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("bs", [32, 64, 128])
def test_decode(bs, D):
    dev = require_gpu()
    S, Hq, Hkv = 333, 8, 2
    print(f"decode token strides block {bs} D={D}", flush=True)
    nb = -(-S // bs)
    q = wl.randn_bf16((1, Hq, 1, D), 81, scale=1.0).to(dev)
    kv = [wl.randn_bf16((1, Hkv, S, D), 82 + i, scale=1.0).to(dev) for i in range(2)]
    mask = torch.ones(1, Hq, 1, nb, dtype=torch.bool, device=dev)
    lens = torch.tensor([S - 3], dtype=torch.int32, device=dev)
    attn = BlockSparseFlashAttention(block_size=bs, min_sparsity_for_speedup=0.0)
    for i in range(2):
        for view in _views(Hkv, S, D, 90 + i, dev):
            t = list(kv)
            t[i] = view
            c = [x.contiguous() for x in t]
            for n in (None, lens):
                assert torch.equal(attn.forward_decode(q, *t, mask, kv_lens=n),
                                   attn.forward_decode(q, *c, mask, kv_lens=n))
    for page in (8, 16, 64):  # page pools [pages, page, Hkv, D], each page one repeated row
        pages = -(-S // page)
        table = torch.randperm(pages, generator=torch.Generator().manual_seed(page)).view(1, -1)
        table = table.to(dev, torch.int32)
        pools = [wl.randn_bf16((pages, page, Hkv, D), 100 + i, scale=1.0).to(dev) for i in range(2)]
        for i in range(2):
            t = list(pools)
            t[i] = pools[i][:, :1].expand(pages, page, Hkv, D)
            c = [x.contiguous() for x in t]
            m = torch.ones(1, Hq, 1, -(-pages * page // bs), dtype=torch.bool, device=dev)
            assert torch.equal(attn.forward_decode_paged(q, *t, table, lens, m),
                               attn.forward_decode_paged(q, *c, table, lens, m))
