"""The work a user of this package has it do, as cases for timing and comparison.

Each case is one call (or one short, self-contained sequence of calls) through the public
entry points: the gate, the block-sparse prefill (dense batch and packed), decode from a
contiguous and from a paged cache, a cached generation through ``SparseAttentionDecoder``
and a gate training step. The geometries are those of ``tasft_amd.workloads`` and
``bench.py`` (Llama-3-8B and Qwen-2.5-7B heads) and generic ones beside them.

``listed()`` names the cases, ``draw(rng)`` makes further ones of the same ranges,
``prepare``/``run`` hold the inputs and make one pass, ``work`` counts the bytes and
operations a pass cannot do without, ``exact`` is the result in 64 bits as plain torch
gives it, and ``tolerance`` how far another correct implementation may be from it.
"""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from tasft_amd.inference import SparseAttentionDecoder
from tasft_amd.kernels import BlockSparseFlashAttention
from tasft_amd.modules import AttnGate
from tasft_amd.training import gate_loss_from_qk

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def listed() -> list[dict]:
    return [
        # The gate over a batch of long prompts before their prefill: the benchmark's
        # geometry (Llama-3-8B heads, trained hidden width 128).
        _gate(name="gate_batch", batch=4, seq=8192),
        # The gate of one short chat prompt, at the default hidden width: launches and host
        # time count. A length that ends inside a block.
        _gate(name="gate_chat", batch=1, seq=1000, hidden=32, dtype="fp16"),
        # Prefill of a batch of long prompts at 80% sparsity (the benchmark's headline).
        _prefill(name="prefill_batch", batch=4, seq=8192, keep=0.2),
        # Prefill of one short prompt.
        _prefill(name="prefill_short", batch=1, seq=2048, keep=0.2),
        # Long-context prefill with a local band, a few global key blocks and the rest at
        # random: Qwen-2.5-7B heads.
        _prefill(name="prefill_long", batch=2, q_heads=28, kv_heads=4, seq=16384, keep=0.25,
                 band=8, sinks=4),
        # A model of head dimension 64 without grouped heads, in fp16, with the finest blocks
        # and a length that ends inside a block.
        _prefill(name="prefill_d64", batch=2, q_heads=16, kv_heads=16, seq=4000, head_dim=64,
                 block=32, keep=0.25, band=2, sinks=1, dtype="fp16"),
        # The prompts of several requests packed into one batch, as a serving engine has them.
        _varlen(name="prefill_packed", lens="8192,6144,4096,2048", keep=0.2),
        # Decode of a large batch over a long contiguous cache, a tenth of the blocks kept.
        _decode(name="decode_batch", batch=64, seq=32768, keep=0.1),
        # Decode of a few requests of different lengths over a paged cache, each query head
        # with its own selection: Qwen-2.5-7B heads.
        _decode(name="decode_paged", batch=8, q_heads=28, kv_heads=4, seq=8192, keep=0.1,
                page=16, shared=False, ragged=True),
        # One short generation through a layer: gate and prefill of the prompt, then cached
        # decode steps, each selecting its key blocks.
        _generate(name="generate", batch=2, seq=2000, steps=16),
        # A gate training step of one layer (forward, target, loss, backward) on full-length
        # sequences.
        _train(name="train_batch", batch=4, seq=8192),
        # The same on a padded batch of shorter examples, at the default hidden width.
        _train(name="train_padded", batch=4, seq=1500, hidden=32, padded=True),
    ]


def draw(rng) -> dict:
    heads, kv = rng.choice([(32, 8), (28, 4), (16, 16), (8, 2), (12, 4)])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    d = rng.choice([128, 128, 64])
    block = rng.choice([64, 64, 32, 128])
    kind = rng.choice(["gate", "prefill", "prefill", "varlen", "decode", "decode", "generate", "train"])
    common = {"q_heads": heads, "kv_heads": kv, "head_dim": d, "block": block, "dtype": dtype}

    def length(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def batch_for(seq, tokens, most=8):
        return rng.randint(1, max(1, min(most, tokens // seq)))

    if kind == "gate":
        seq = length(100, 8192)
        return _gate(batch=batch_for(seq, 32768), seq=seq, hidden=rng.choice([32, 64, 128]), **common)
    if kind == "prefill":
        longest = 16384 if block > 32 else 8192
        seq = length(100, longest)
        return _prefill(batch=batch_for(seq, longest), seq=seq, keep=round(rng.uniform(0.05, 0.3), 3),
                        band=rng.choice([1, 1, 2, 8]), sinks=rng.choice([0, 1, 4]),
                        causal=seq > 4096 or rng.random() < 0.8, **common)
    if kind == "varlen":
        left, lens = 16384 if block > 32 else 8192, []
        for _ in range(rng.randint(2, 8)):
            n = length(50, min(8192, left))
            lens.append(n)
            left -= n
            if left < 100:
                break
        return _varlen(lens=",".join(str(n) for n in lens), keep=round(rng.uniform(0.1, 0.3), 3), **common)
    if kind == "decode":
        seq = length(256, 32768)
        return _decode(batch=batch_for(seq, 64 * 8192, 64), seq=seq, keep=round(rng.uniform(0.05, 0.4), 3),
                       page=rng.choice([0, 16, 32, 64]), shared=rng.random() < 0.5,
                       ragged=rng.random() < 0.5, **common)
    if kind == "generate":
        seq = length(100, 4096)
        return _generate(batch=batch_for(seq, 8192, 4), seq=seq, steps=rng.randint(4, 24),
                         hidden=rng.choice([32, 64, 128]), **common)
    seq = length(200, 4096)
    return _train(batch=batch_for(seq, 8192, 4), seq=seq, hidden=rng.choice([32, 64, 128]),
                  padded=rng.random() < 0.5, **common)


# ---------------------------------------------------------------------- case constructors
def _case(kind, name, **fields):
    case = {"kind": kind, "q_heads": 32, "kv_heads": 8, "head_dim": 128, "block": 64, "dtype": "bf16"}
    case.update(fields)
    if name is not None:
        case["name"] = name
    return case


def _gate(name=None, hidden=128, keep=0.2, **f):
    return _case("gate", name, hidden=hidden, keep=keep, **f)


def _prefill(name=None, band=1, sinks=0, causal=True, **f):
    return _case("prefill", name, band=band, sinks=sinks, causal=causal, **f)


def _varlen(name=None, **f):
    return _case("varlen", name, **f)


def _decode(name=None, page=0, shared=True, ragged=False, **f):
    return _case("decode", name, page=page, shared=shared, ragged=ragged, **f)


def _generate(name=None, hidden=128, keep=0.2, **f):
    return _case("generate", name, hidden=hidden, keep=keep, **f)


def _train(name=None, hidden=128, padded=False, **f):
    return _case("train", name, hidden=hidden, padded=padded, **f)


# ------------------------------------------------------------------------------- inputs
def _generator(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, shape, dtype):
    return torch.randn(shape, generator=g, device="cuda", dtype=dtype)


def _projected(g, shape, dtype, period=64):
    """Queries or keys as a layer projects them: unit-scale noise around a component that
    changes every ``period`` tokens, so that the block means (what the gate sees) spread.
    ``shape`` is [B, H, S, D]."""
    b, h, s, d = shape
    x = _randn(g, shape, dtype)
    topic = _randn(g, (b, h, -(-s // period), d), dtype) * 0.5
    return x.add_(topic.repeat_interleave(period, dim=2)[:, :, :s])


def _make_gate(case, g):
    """A gate as training leaves it: the input projection at its initial scale, biases and
    an output layer whose logits spread over a few tenths."""
    gate = AttnGate(num_heads=case["q_heads"], head_dim=case["head_dim"], block_size=case["block"],
                    gate_hidden_dim=case["hidden"]).to("cuda")
    with torch.no_grad():
        w = gate.gate_proj_in.weight
        bound = math.sqrt(6.0 / (w.shape[0] + w.shape[1]))
        w.copy_((torch.rand(w.shape, generator=g, device="cuda") * 2 - 1) * bound)
        gate.gate_proj_in.bias.copy_(_randn(g, w.shape[:1], torch.float32) * 0.05)
        gate.gate_proj_out.weight.copy_(_randn(g, (1, w.shape[0]), torch.float32) * 0.3)
    return gate


def _pool(x, block):
    pad = -x.shape[2] % block
    x = F.pad(x, (0, 0, 0, pad)) if pad else x
    return x.view(x.shape[0], x.shape[1], -1, block, x.shape[3]).sum(3) / block


def _gate_scores(q, k, w_in, b_in, w_out, block, dt):
    """The gate's soft scores of one batch entry (causal zeros included), in ``dt``."""
    d = q.shape[-1]
    qb, kb = _pool(q.to(dt), block), _pool(k.to(dt), block)
    uq = qb @ w_in[:, :d].t() + b_in
    uk = (kb @ w_in[:, d:].t()).repeat_interleave(q.shape[1] // k.shape[1], dim=1)
    logits = F.relu(uq.unsqueeze(3) + uk.unsqueeze(2)) @ w_out.reshape(-1)
    return torch.sigmoid(logits).tril()


def _gate_weights(gate, dt):
    return (gate.gate_proj_in.weight.detach().to(dt), gate.gate_proj_in.bias.detach().to(dt),
            gate.gate_proj_out.weight.detach().to(dt))


def _calibrate(gate, q, k, keep):
    """Per-head thresholds that keep about ``keep`` of the causal blocks of the first
    sequence, halfway between two neighbouring scores."""
    soft = _gate_scores(q[:1], k[:1], *_gate_weights(gate, torch.float32), gate.block_size, torch.float32)[0]
    nb = soft.shape[-1]
    causal = torch.ones(nb, nb, dtype=torch.bool, device="cuda").tril()
    vals = soft[:, causal].sort(dim=1, descending=True).values
    n = min(max(1, round(keep * vals.shape[1])), vals.shape[1] - 1)
    if n < 1:
        return torch.full((soft.shape[0],), 0.5, device="cuda")
    return (vals[:, n - 1] + vals[:, n]) / 2


def _block_mask(case, g, batch, nb):
    """[batch, Hq, nb, nb] bool: a band of ``band`` blocks along the diagonal, ``sinks``
    leading key blocks, and each other block with probability ``keep``."""
    i = torch.arange(nb, device="cuda")
    near = (i[:, None] - i[None, :]).abs() < case.get("band", 1)
    fixed = near | (i[None, :] < case.get("sinks", 0))
    rand = torch.rand((batch, case["q_heads"], nb, nb), generator=g, device="cuda") < case["keep"]
    m = rand | fixed
    return m.tril() if case.get("causal", True) else m


def _lens(case):
    return [int(n) for n in case["lens"].split(",")]


def prepare(case: dict, seed: int) -> dict:
    g = _generator(seed)
    kind, dt = case["kind"], _DTYPES[case["dtype"]]
    hq, hkv, d, bs = case["q_heads"], case["kv_heads"], case["head_dim"], case["block"]
    st = {"case": case}
    if kind == "gate":
        b, s = case["batch"], case["seq"]
        st["q"] = _projected(g, (b, hq, s, d), dt)
        st["k"] = _projected(g, (b, hkv, s, d), dt)
        st["gate"] = _make_gate(case, g).requires_grad_(False)
        st["taus"] = _calibrate(st["gate"], st["q"], st["k"], case["keep"])
    elif kind == "prefill":
        b, s = case["batch"], case["seq"]
        st["q"] = _projected(g, (b, hq, s, d), dt)
        st["k"] = _projected(g, (b, hkv, s, d), dt)
        st["v"] = _randn(g, (b, hkv, s, d), dt)
        st["mask"] = _block_mask(case, g, b, -(-s // bs))
        st["attn"] = BlockSparseFlashAttention(block_size=bs, min_sparsity_for_speedup=0.0)
    elif kind == "varlen":
        lens = _lens(case)
        t = sum(lens)
        st["q"] = _projected(g, (1, hq, t, d), dt)[0].transpose(0, 1).contiguous()
        st["k"] = _projected(g, (1, hkv, t, d), dt)[0].transpose(0, 1).contiguous()
        st["v"] = _randn(g, (t, hkv, d), dt)
        st["mask"] = _block_mask(case, g, len(lens), -(-max(lens) // bs))
        st["cu"] = torch.tensor([0] + lens, device="cuda").cumsum(0).to(torch.int32)
        st["attn"] = BlockSparseFlashAttention(block_size=bs, min_sparsity_for_speedup=0.0)
    elif kind == "decode":
        b, s, page = case["batch"], case["seq"], case["page"]
        if page:
            s = -(-s // page) * page
        nb = -(-s // bs)
        st["q"] = _randn(g, (b, hq, 1, d), dt)
        lens = torch.full((b,), s, dtype=torch.int32, device="cuda")
        if case["ragged"]:
            lens = torch.randint(s // 2, s + 1, (b,), generator=g, device="cuda", dtype=torch.int32)
        # The first block and the newest one are always selected, as a sparse decode keeps them.
        h = hkv if case["shared"] else hq
        m = torch.rand((b, h, 1, nb), generator=g, device="cuda") < case["keep"]
        j = torch.arange(nb, device="cuda")
        newest = ((lens - 1) // bs).view(b, 1, 1, 1)
        m = ((m | (j == 0)) & (j < newest)) | (j == newest)
        st["mask"] = m.repeat_interleave(hq // h, dim=1)
        if page:
            per = s // page
            perm = torch.randperm(b * per, generator=g, device="cuda")
            st["table"] = perm.view(b, per).to(torch.int32)
            st["k"] = _randn(g, (b * per, page, hkv, d), dt)
            st["v"] = _randn(g, (b * per, page, hkv, d), dt)
            st["lens"] = lens
        else:
            st["k"] = _randn(g, (b, hkv, s, d), dt)
            st["v"] = _randn(g, (b, hkv, s, d), dt)
            st["lens"] = lens if case["ragged"] else None
        st["attn"] = BlockSparseFlashAttention(block_size=bs, min_sparsity_for_speedup=0.0)
    elif kind == "generate":
        b, s, n = case["batch"], case["seq"], case["steps"]
        st["q"] = _projected(g, (b, hq, s + n, d), dt)
        st["k"] = _projected(g, (b, hkv, s + n, d), dt)
        st["v"] = _randn(g, (b, hkv, s + n, d), dt)
        gate = _make_gate(case, g).requires_grad_(False)
        st["taus"] = _calibrate(gate, st["q"][:, :, :s], st["k"][:, :, :s], case["keep"])
        st["gate"] = gate
        st["prompt"] = tuple(st[x][:, :, :s].contiguous() for x in "qkv")
        st["new_q"] = [st["q"][:, :, s + t:s + t + 1].contiguous() for t in range(n)]
        st["decoder"] = SparseAttentionDecoder(gate, threshold=st["taus"], max_len=s + n)
    else:
        b, s = case["batch"], case["seq"]
        st["q"] = _projected(g, (b, hq, s, d), dt)
        st["k"] = _projected(g, (b, hkv, s, d), dt)
        st["gate"] = _make_gate(case, g)
        st["pad"] = None
        if case["padded"]:
            # A key-padding row per sequence, additive, at the masking value HF models use.
            lens = torch.randint(s // 2, s + 1, (b,), generator=g, device="cuda")
            lens[0] = s
            dead = torch.arange(s, device="cuda")[None, :] >= lens[:, None]
            st["pad"] = torch.zeros((b, s), device="cuda").masked_fill(dead, torch.finfo(torch.float32).min)
    return st


def run(st: dict):
    kind = st["case"]["kind"]
    if kind == "gate":
        out = st["gate"](st["q"], st["k"], threshold=st["taus"], force_diagonal=True)
        return {"soft": out.soft_scores, "mask": out.hard_mask}
    if kind == "prefill":
        return st["attn"].forward(st["q"], st["k"], st["v"], st["mask"], causal=st["case"]["causal"])
    if kind == "varlen":
        return st["attn"].forward_varlen(st["q"], st["k"], st["v"], st["mask"], st["cu"],
                                         max_seqlen=max(_lens(st["case"])))
    if kind == "decode":
        if st["case"]["page"]:
            return st["attn"].forward_decode_paged(st["q"], st["k"], st["v"], st["table"], st["lens"],
                                                   st["mask"])
        return st["attn"].forward_decode(st["q"], st["k"], st["v"], st["mask"], kv_lens=st["lens"])
    if kind == "generate":
        dec, s = st["decoder"], st["case"]["seq"]
        out, gate_out = dec.prefill(*st["prompt"])
        outs, rows = [], []
        for t, q_new in enumerate(st["new_q"]):
            o, row = dec.step(q_new, st["k"][:, :, :s + t + 1], st["v"][:, :, :s + t + 1])
            outs.append(o)
            rows.append(row.soft_scores)
        return {"prompt": out, "prompt_soft": gate_out.soft_scores, "steps": outs, "rows": rows}
    gate = st["gate"]
    gate.zero_grad(set_to_none=True)
    out = gate(st["q"], st["k"])
    loss = gate_loss_from_qk(out.soft_scores, st["q"], st["k"], st["case"]["block"],
                             attention_mask=st["pad"])
    loss.backward()
    return {"loss": loss.detach(), "w_in": gate.gate_proj_in.weight.grad,
            "b_in": gate.gate_proj_in.bias.grad, "w_out": gate.gate_proj_out.weight.grad}


# --------------------------------------------------------------------------------- work
def _pairs(seq, block, keep, band, sinks, causal):
    """Expected (query, key) token pairs of one head's block mask."""
    nb = -(-seq // block)
    total = 0.0
    for i in range(nb):
        rows = min(block, seq - i * block)
        near = min(i, band - 1)  # full blocks of the band left of the diagonal
        far = i - near
        sink = min(sinks, far)
        left = near + sink + keep * (far - sink)
        total += rows * block * left + (rows * (rows + 1) / 2 if causal else rows * rows)
        if not causal:
            right = nb - 1 - i
            fixed = max(min(right, band - 1), min(right, max(0, sinks - 1 - i)))
            total += rows * block * (fixed + keep * (right - fixed))
    return total


def work(case: dict) -> dict:
    kind = case["kind"]
    hq, hkv, d, bs = case["q_heads"], case["kv_heads"], case["head_dim"], case["block"]
    if kind in ("gate", "train", "generate"):
        b, s, hid = case["batch"], case["seq"], case["hidden"]
        nb = -(-s // bs)
        blocks = b * (hq + hkv) * nb
        pairs = b * hq * nb * (nb + 1) / 2
        qk = b * (hq + hkv) * s * d * 2
        pool = b * (hq + hkv) * s * d + 2 * blocks * d * hid
        mlp = 3 * pairs * hid
    if kind == "gate":
        return {"bytes": qk + b * hq * nb * nb * 5 + hid * (2 * d + 2) * 4, "flops": pool + mlp}
    if kind == "train":
        # Scores of every causal pair for the target, and the gate's backward: two sums
        # per pair and unit, then the weight gradients.
        scores = 2.0 * b * hq * d * s * (s + 1) / 2
        back = 4 * pairs * hid + 2 * blocks * d * hid
        return {"bytes": qk + hid * (2 * d + 2) * 8, "flops": scores + pool + mlp + back}
    if kind == "prefill":
        b, s = case["batch"], case["seq"]
        nb = -(-s // bs)
        pairs = b * hq * _pairs(s, bs, case["keep"], case["band"], case["sinks"], case["causal"])
        return {"bytes": 2 * b * (hq + hkv) * s * d * 2 + b * hq * nb * nb, "flops": 4 * d * pairs}
    if kind == "varlen":
        lens = _lens(case)
        pairs = hq * sum(_pairs(n, bs, case["keep"], 1, 0, True) for n in lens)
        nbytes = 2 * sum(lens) * (hq + hkv) * d * 2 + hq * sum((-(-n // bs)) ** 2 for n in lens)
        return {"bytes": nbytes, "flops": 4 * d * pairs}
    if kind == "decode":
        b, s = case["batch"], case["seq"]
        mean = 0.75 * s if case["ragged"] else s
        nb = -(-s // bs)
        union = case["keep"] if case["shared"] else 1 - (1 - case["keep"]) ** (hq // hkv)
        tokens = min(mean, 2 * bs + union * max(0.0, mean - 2 * bs))
        own = min(mean, 2 * bs + case["keep"] * max(0.0, mean - 2 * bs))
        return {"bytes": b * hkv * tokens * d * 4 + 2 * b * hq * d * 2 + b * hq * nb,
                "flops": 4 * b * hq * d * own}
    n = case["steps"]
    prompt = b * hq * _pairs(s, bs, case["keep"], 1, 0, True)
    selected = bs + case["keep"] * s
    union = min(s, bs + (1 - (1 - case["keep"]) ** (hq // hkv)) * s)
    return {"bytes": 2 * qk + b * hq * nb * nb * 4 + n * b * hkv * union * d * 4,
            "flops": pool + mlp + 4 * d * prompt + n * (4 * b * hq * d * selected + 3 * b * hq * nb * hid)}


# --------------------------------------------------------------------------- comparison
def tolerance(case: dict) -> dict:
    # About four times the error against 64 bits that the path shows (in brackets).
    kind, half = case["kind"], case["dtype"] == "fp16"
    if kind == "gate":
        # fp32 sums of 16-bit inputs, a sigmoid (2e-7); a mask bit may fall either way at a
        # score within rounding of its threshold.
        return {"rel": 1e-6, "differ": 1e-4}
    if kind == "train":
        # fp32 sums behind a ReLU (2.4e-5): a unit within rounding of zero counts or not.
        return {"rel": 1e-4}
    if kind == "generate":
        # As attention, and a key block whose score is within rounding of its threshold may
        # be selected or not.
        return {"rel": 2e-3 if half else 1e-2}
    # Probabilities and output rounded to 16 bits, fp32 sums (2.2e-3, in fp16 2.5e-4).
    return {"rel": 1e-3 if half else 8e-3}


def _attention64(q, k, v, mask, block, causal):
    """Block-sparse attention of [B, H, S, D] inputs in 64 bits, head by head."""
    b, hq, s, d = q.shape
    grp = hq // k.shape[1]
    out = torch.zeros((b, hq, s, d), dtype=torch.float64, device=q.device)
    pos = torch.arange(s, device=q.device)
    step = max(block, (1 << 25) // s // block * block)
    for i in range(b):
        for h in range(hq):
            kk, vv = k[i, h // grp].double(), v[i, h // grp].double()
            for r in range(0, s, step):
                e = min(s, r + step)
                c = e if causal else s  # no key past the chunk's last row
                scores = (q[i, h, r:e].double() @ kk[:c].t()) * (1.0 / math.sqrt(d))
                m = mask[i, h, pos[r:e] // block][:, pos[:c] // block] != 0
                if causal:
                    m &= pos[None, :c] <= pos[r:e, None]
                p = torch.softmax(scores.masked_fill_(~m, -math.inf), dim=-1).nan_to_num_(0.0)
                out[i, h, r:e] = p @ vv[:c]
    return out


def _decode64(q, k, v, mask, lens, block):
    """One query per head over [B, Hkv, S, D] caches in 64 bits; ``mask`` [B, Hq, 1, NB]."""
    b, hq, _, d = q.shape
    grp = hq // k.shape[1]
    s = k.shape[2]
    pos = torch.arange(s, device=q.device)
    out = []
    for i in range(b):
        kk = k[i].double().repeat_interleave(grp, 0)
        vv = v[i].double().repeat_interleave(grp, 0)
        m = mask[i][:, :, pos // block] & (pos < int(lens[i]))
        scores = (q[i].double() @ kk.transpose(1, 2).contiguous()) / math.sqrt(d)
        p = torch.softmax(scores.masked_fill(~m, -math.inf), dim=-1).nan_to_num(0.0)
        out.append(p @ vv)
    return torch.stack(out)


def _target64(q, k, block, pad):
    """Flat softmax of the block maxima of the causal scores of one sequence, per head."""
    h, s, d = q.shape
    grp = h // k.shape[0]
    nb = -(-s // block)
    tail = nb * block - s
    pos = torch.arange(s, device=q.device)
    step = max(block, (1 << 25) // s // block * block)
    out = []
    for i in range(h):
        kk = k[i // grp].double()
        rows = []
        for r in range(0, s, step):
            e = min(s, r + step)
            sc = (q[i, r:e].double() @ kk.t()) / math.sqrt(d)
            sc.masked_fill_(pos[None, :] > pos[r:e, None], -math.inf)
            if pad is not None:
                sc += pad
            sc = F.pad(sc, (0, tail, 0, -(e - r) % block), value=-math.inf)
            rows.append(sc.view(sc.shape[0] // block, block, nb, block).amax((1, 3)))
        out.append(torch.softmax(torch.cat(rows).view(-1), 0).view(nb, nb))
    return torch.stack(out)


def exact(case: dict, seed: int):
    st = prepare(case, seed)
    kind, bs = case["kind"], case["block"]
    if kind == "gate":
        w = _gate_weights(st["gate"], torch.float64)
        soft = torch.cat([_gate_scores(st["q"][i:i + 1], st["k"][i:i + 1], *w, bs, torch.float64)
                          for i in range(case["batch"])])
        nb = soft.shape[-1]
        mask = soft >= st["taus"].double().view(1, -1, 1, 1)
        return {"soft": soft, "mask": mask | torch.eye(nb, dtype=torch.bool, device="cuda")}
    if kind == "prefill":
        return _attention64(st["q"], st["k"], st["v"], st["mask"], bs, case["causal"])
    if kind == "varlen":
        outs, start = [], 0
        for i, n in enumerate(_lens(case)):
            q, k, v = (st[x][start:start + n].transpose(0, 1).unsqueeze(0) for x in "qkv")
            nb = -(-n // bs)
            outs.append(_attention64(q, k, v, st["mask"][i:i + 1, :, :nb, :nb], bs, True)[0].transpose(0, 1))
            start += n
        return torch.cat(outs)
    if kind == "decode":
        k, v, b = st["k"], st["v"], case["batch"]
        if case["page"]:
            t = st["table"].long()
            k, v = (x[t].flatten(1, 2).transpose(1, 2) for x in (k, v))
        lens = st["lens"] if st["lens"] is not None else [k.shape[2]] * b
        return _decode64(st["q"], k, v, st["mask"], lens, bs)
    if kind == "generate":
        s, n = case["seq"], case["steps"]
        w = _gate_weights(st["gate"], torch.float64)
        taus = st["taus"].double().view(1, -1, 1, 1)
        q, k, v = st["q"], st["k"], st["v"]
        soft = torch.cat([_gate_scores(q[i:i + 1, :, :s], k[i:i + 1, :, :s], *w, bs, torch.float64)
                          for i in range(case["batch"])])
        eye = torch.eye(soft.shape[-1], dtype=torch.bool, device="cuda")
        prompt = _attention64(*st["prompt"], (soft >= taus) | eye, bs, True)
        outs, rows = [], []
        for t in range(s, s + n):
            # The step's row is the last row of the gate on the sequence so far.
            full = torch.cat([_gate_scores(q[i:i + 1, :, :t + 1], k[i:i + 1, :, :t + 1], *w, bs,
                                           torch.float64)[:, :, -1:] for i in range(case["batch"])])
            m = full >= taus
            m[..., -1] = True
            rows.append(full)
            outs.append(_decode64(q[:, :, t:t + 1], k[:, :, :t + 1], v[:, :, :t + 1], m,
                                  [t + 1] * case["batch"], bs))
        return {"prompt": prompt, "prompt_soft": soft, "steps": outs, "rows": rows}
    eps = 1e-8
    params = [w.requires_grad_(True) for w in _gate_weights(st["gate"], torch.float64)]
    total = 0.0
    for i in range(case["batch"]):
        pad = None if st["pad"] is None else st["pad"][i].double()
        target = _target64(st["q"][i], st["k"][i], bs, pad)
        soft = _gate_scores(st["q"][i:i + 1], st["k"][i:i + 1], *params, bs, torch.float64)[0]
        soft, target = soft.flatten(1), target.flatten(1)
        dist = soft / (soft.sum(-1, keepdim=True) + eps)
        loss = F.kl_div(torch.log(dist + eps), target, reduction="sum") / case["batch"]
        loss.backward()
        total = total + loss.detach()
    return {"loss": total, "w_in": params[0].grad, "b_in": params[1].grad, "w_out": params[2].grad}
