"""The work whose time is tracked: calls of the public ops over the range a transformer program makes.

A case is one op (`op`), its sizes, its dtype and its direction: `train` False is the call without a
graph, True is the call and its gradients through autograd. `listed()` holds fixed cases, `draw(rng)`
gives more of the same ranges:

    rms_norm, add_rms_norm    1 to 65536 rows of 64 to 8192 columns
    swiglu                    1 to 16384 rows of 64 to 14336 columns, gate and up separate or fused
    rotary_embedding, rope,   1 to 16 sequences of 1 to 8192 positions, 1 to 64 heads
    qk_norm_rope
    attn, attn_varlen         2 to 16384 tokens, 1 to 64 heads in groups of 1 to 8, head_dim 16 to 256

`prepare` makes the tensors of one pass from a seed, `run` is the pass, `work` the bytes and operations
it cannot do without, `tolerance` what two correct implementations may differ by, and `exact` the same
outputs from float64 torch.
"""

from __future__ import annotations

import math
import random

import torch

from popcorn_amd import impls

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
THETA = 500000.0
EPS = 1e-6


def listed() -> list[dict]:
    return [
        # one decode step of a batch of 16 requests: the residual add and norm in front of a block
        {"name": "decode_add_norm", "op": "add_rms_norm", "rows": 16, "cols": 4096, "dtype": "bf16", "wide_weight": False,
         "offset": 0.0, "train": False},
        # a training micro-batch of 8192 tokens through a norm
        {"name": "norm_train", "op": "rms_norm", "rows": 8192, "cols": 4096, "dtype": "bf16", "wide_weight": False,
         "bias": False, "train": True},
        # an odd width, as in a small head or a concatenated feature, in fp32 with a bias
        {"name": "norm_odd_train", "op": "rms_norm", "rows": 5003, "cols": 1537, "dtype": "fp32", "wide_weight": False,
         "bias": True, "train": True},
        # the pre-norm residual stream of a large layer under autocast (fp32 weight beside 16-bit activations)
        {"name": "add_norm_autocast_train", "op": "add_rms_norm", "rows": 16384, "cols": 8192, "dtype": "bf16",
         "wide_weight": True, "offset": 1.0, "train": True},
        # the MLP gate of a layer whose gate and up projections are one matrix product: two halves of its output
        {"name": "swiglu_fused_train", "op": "swiglu", "rows": 8192, "cols": 14336, "dtype": "bf16", "fused": True,
         "train": True},
        # rotary embedding of the q and k views of a packed qkv projection, in prefill
        {"name": "rotary_packed", "op": "rotary_embedding", "batch": 2, "seq": 4096, "q_heads": 32, "kv_heads": 8,
         "head_dim": 128, "half": 64, "dtype": "bf16", "tables": "fp32", "interleaved": False, "train": False},
        # the q/k norm and rope of a training layer, [batch, seq, heads, dim] projections viewed heads-first
        {"name": "qk_norm_rope_train", "op": "qk_norm_rope", "batch": 2, "seq": 4096, "q_heads": 32, "kv_heads": 8,
         "head_dim": 128, "dtype": "bf16", "tables": "bf16", "train": True},
        # the prompt of one request: short, of no round length
        {"name": "attn_prefill", "op": "attn", "batch": 1, "seq": 1021, "q_heads": 32, "kv_heads": 8, "head_dim": 128,
         "dtype": "bf16", "causal": True, "train": False},
        # long-context training of one sequence on a shard of the heads (one kv head's group on a device)
        {"name": "attn_long_shard_train", "op": "attn", "batch": 1, "seq": 16384, "q_heads": 4, "kv_heads": 1,
         "head_dim": 128, "dtype": "bf16", "causal": True, "train": True},
        # a training layer at the benchmark's attention shape
        {"name": "attn_train", "op": "attn", "batch": 4, "seq": 8192, "q_heads": 32, "kv_heads": 8, "head_dim": 128,
         "dtype": "bf16", "causal": True, "train": True},
        # packed documents of very different lengths, one kv head per q head
        {"name": "attn_packed_train", "op": "attn_varlen", "total": 16384, "segments": 23, "q_heads": 16, "kv_heads": 16,
         "head_dim": 64, "dtype": "bf16", "causal": True, "train": True},
        # an encoder over patches plus one class token: full attention in fp16
        {"name": "attn_encoder_train", "op": "attn", "batch": 8, "seq": 1025, "q_heads": 12, "kv_heads": 12, "head_dim": 64,
         "dtype": "fp16", "causal": False, "train": True},
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    """An integer of [lo, hi], even over the logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def _width(rng: random.Random, lo: int, hi: int) -> int:
    """A row width: mostly whole 64s, as models have them, else any integer."""
    n = _log_int(rng, lo, hi)
    return max(lo, n // 64 * 64) if rng.random() < 0.7 else n


def _dtype(rng: random.Random) -> str:
    return rng.choices(("bf16", "fp16", "fp32"), (5, 2, 2))[0]


def draw(rng: random.Random) -> dict:
    op = rng.choice(("rms_norm", "add_rms_norm", "swiglu", "rotary_embedding", "rope", "qk_norm_rope", "attn", "attn",
                     "attn_varlen"))
    case: dict = {"op": op, "dtype": _dtype(rng), "train": rng.random() < 0.6}
    if op in ("rms_norm", "add_rms_norm"):
        cols = _width(rng, 64, 8192)
        case.update(rows=_log_int(rng, 1, min(65536, (1 << 28) // cols)), cols=cols,
                    wide_weight=case["dtype"] != "fp32" and rng.random() < 0.25)
        case.update({"bias": rng.random() < 0.25} if op == "rms_norm" else {"offset": rng.choice((0.0, 1.0))})
        return case
    if op == "swiglu":
        case.update(rows=_log_int(rng, 1, 16384), cols=_width(rng, 64, 14336), fused=rng.random() < 0.5)
        return case
    group = rng.choice((1, 1, 2, 3, 4, 4, 5, 8))
    kv_heads = _log_int(rng, 1, 64 // group)
    case.update(q_heads=kv_heads * group, kv_heads=kv_heads)
    if op in ("rotary_embedding", "rope", "qk_norm_rope"):
        dims = (32, 64, 64, 128, 128, 256) if op == "qk_norm_rope" else (32, 64, 80, 96, 128, 128, 192, 256)
        head_dim = rng.choice(dims)
        case.update(head_dim=head_dim, batch=_log_int(rng, 1, 16),
                    tables="fp32" if case["dtype"] == "fp32" else rng.choice((case["dtype"], "fp32")))
        row = case["batch"] * (kv_heads * group + kv_heads) * head_dim
        case["seq"] = _log_int(rng, 1, max(1, min(8192, (1 << 27) // row)))
        if op == "rotary_embedding":
            case.update(half=rng.choice((head_dim // 2, head_dim // 2, head_dim // 4)), interleaved=rng.random() < 0.3)
        return case
    head_dim = rng.choice((16, 32, 64, 64, 64, 80, 96, 128, 128, 128, 192, 256))
    case.update(head_dim=head_dim, causal=rng.random() < 0.7)
    # at most about a tenth of the largest listed case's operations, a 160th in fp32 (a sixteenth of the rate)
    ops = 7e11 if case["dtype"] != "fp32" else 4.5e10
    per_pair = 4 * head_dim * case["q_heads"] * (3.5 if case["train"] else 1.0)
    longest = int(math.sqrt(ops / per_pair))
    if op == "attn":
        case["seq"] = _log_int(rng, 2, min(16384, longest))  # a lone token has no gradient of its scores to compare
        case["batch"] = _log_int(rng, 1, max(1, min(16, 16384 // case["seq"], int((longest / case["seq"]) ** 2))))
    else:
        case["segments"] = _log_int(rng, 1, 64)
        case["total"] = _log_int(rng, 2 * case["segments"], max(2 * case["segments"], min(16384, longest)))
    return case


# ------------------------------------------------------------------ inputs


def _lengths(total: int, segments: int) -> list[int]:
    """Document lengths of a packed batch, spread over their logarithm (a fixed order, short and long mixed)."""
    order = random.Random(segments)
    weights = [math.exp(order.uniform(0.0, math.log(100.0))) for _ in range(segments)]
    scale = (total - segments) / sum(weights)
    lengths = [1 + int(w * scale) for w in weights]
    lengths[-1] += total - sum(lengths)
    return lengths


def _angles(seq: int, half: int, dev: torch.device) -> torch.Tensor:
    freq = THETA ** (-torch.arange(half, device=dev, dtype=torch.float64) / half)
    return torch.arange(seq, device=dev, dtype=torch.float64)[:, None] * freq


def prepare(case: dict, seed: int) -> dict:
    dev = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=dev).manual_seed(seed)
    dtype, op, train = DTYPES[case["dtype"]], case["op"], case["train"]

    def randn(*shape, dt=dtype):
        return torch.randn(shape, generator=gen, device=dev, dtype=torch.float32).to(dt)

    def scale_vector(n, dt):
        return (1.0 + 0.1 * torch.randn(n, generator=gen, device=dev)).to(dt)

    state = {"case": case}
    if op in ("rms_norm", "add_rms_norm"):
        rows, cols = case["rows"], case["cols"]
        wdt = torch.float32 if case["wide_weight"] else dtype
        state["x"] = randn(rows, cols)
        if op == "add_rms_norm":
            state["residual"] = randn(rows, cols)
            # the offset form keeps its weight around zero
            state["weight"] = (scale_vector(cols, torch.float32) - case["offset"]).to(wdt)
            inputs, cotangents = ("x", "residual", "weight"), ((rows, cols, wdt), (rows, cols, dtype))
        else:
            state["weight"] = scale_vector(cols, wdt)
            state["bias"] = randn(cols, dt=wdt) if case["bias"] else None
            inputs = ("x", "weight", "bias") if case["bias"] else ("x", "weight")
            cotangents = ((rows, cols, wdt),)
        state["dy"] = tuple(randn(r, c, dt=dt) for r, c, dt in cotangents) if train else ()
    elif op == "swiglu":
        rows, cols = case["rows"], case["cols"]
        if case["fused"]:
            state["a"], state["b"] = randn(rows, 2 * cols).chunk(2, dim=-1)
        else:
            state["a"], state["b"] = randn(rows, cols), randn(rows, cols)
        inputs = ("a", "b")
        state["dy"] = (randn(rows, cols),) if train else ()
    elif op in ("rotary_embedding", "rope", "qk_norm_rope"):
        b, s, hq, hkv, d = (case[k] for k in ("batch", "seq", "q_heads", "kv_heads", "head_dim"))
        tdt = DTYPES[case["tables"]]
        qkv = randn(b, s, hq + 2 * hkv, d)  # a packed projection; q and k are views of it
        q, k = qkv[:, :, :hq], qkv[:, :, hq:hq + hkv]
        if op == "rotary_embedding":
            angles = _angles(s, case["half"], dev)
            state["cos"], state["sin"] = angles.cos().to(tdt), angles.sin().to(tdt)
            out = dtype
        else:
            q, k = q.transpose(1, 2), k.transpose(1, 2)
            angles = _angles(s, d // 2, dev).repeat(1, 2)[None]
            state["cos"], state["sin"] = angles.cos().to(tdt), angles.sin().to(tdt)
            out = torch.promote_types(dtype, tdt)
        state["q"], state["k"] = q, k
        inputs = ("q", "k")
        if op == "qk_norm_rope":
            state["q_weight"], state["k_weight"] = scale_vector(d, dtype), scale_vector(d, dtype)
            inputs = ("q", "k", "q_weight", "k_weight")
        state["dy"] = tuple(randn(*t.shape, dt=out) for t in (q, k)) if train else ()
    else:
        hq, hkv, d = case["q_heads"], case["kv_heads"], case["head_dim"]
        lead = (case["batch"], case["seq"]) if op == "attn" else (case["total"],)
        state["q"], state["k"], state["v"] = randn(*lead, hq, d), randn(*lead, hkv, d), randn(*lead, hkv, d)
        if op == "attn_varlen":
            cuts = [0]
            for n in _lengths(case["total"], case["segments"]):
                cuts.append(cuts[-1] + n)
            state["cu_seqlens"] = torch.tensor(cuts, dtype=torch.int32, device=dev)
        inputs = ("q", "k", "v")
        state["dy"] = (randn(*lead, hq, d),) if train else ()
    if train:
        for name in inputs:
            state[name] = state[name].detach().requires_grad_()
        state["inputs"] = tuple(state[name] for name in inputs)
    return state


def run(state: dict):
    case, op = state["case"], state["case"]["op"]
    if op == "rms_norm":
        out = (impls.rms_norm(state["x"], state["weight"], state["bias"], EPS),)
    elif op == "add_rms_norm":
        out = impls.add_rms_norm(state["x"], state["residual"], state["weight"], EPS, case["offset"])
    elif op == "swiglu":
        out = (impls.swiglu(state["a"], state["b"]),)
    elif op == "rotary_embedding":
        out = tuple(impls.rotary_embedding(state[n], state["cos"], state["sin"], case["interleaved"]) for n in ("q", "k"))
    elif op == "rope":
        out = impls.rope(state["q"], state["k"], state["cos"], state["sin"])
    elif op == "qk_norm_rope":
        out = impls.qk_norm_rope(state["q"], state["k"], state["q_weight"], state["k_weight"], state["cos"], state["sin"],
                                 EPS)
    elif op == "attn":
        out = (impls.attn(state["q"], state["k"], state["v"], case["causal"]),)
    else:
        out = (impls.attn_varlen(state["q"], state["k"], state["v"], state["cu_seqlens"], case["causal"]),)
    if not case["train"]:
        return out
    grads = torch.autograd.grad(out, state["inputs"], state["dy"])
    return tuple(t.detach() for t in out) + tuple(grads)


# ------------------------------------------------------------------ what a pass cannot do without


def _pairs(case: dict) -> int:
    """(query, key) pairs of one head."""
    lengths = [case["seq"]] * case["batch"] if case["op"] == "attn" else _lengths(case["total"], case["segments"])
    return sum(n * (n + 1) // 2 if case["causal"] else n * n for n in lengths)


def work(case: dict) -> dict:
    """Bytes of the call's inputs and outputs, and with gradients those of the backward call as well (it comes after the
    whole forward of a program: what it reads, it reads again); matrix operations for attention, five to an element or
    more elsewhere."""
    op, train = case["op"], case["train"]
    e = 4 if case["dtype"] == "fp32" else 2
    if op in ("rms_norm", "add_rms_norm"):
        n, cols = case["rows"] * case["cols"], case["cols"]
        ew = 4 if case["wide_weight"] else e
        vectors = (2 if case.get("bias") else 1) * cols * ew
        add = op == "add_rms_norm"
        fwd = n * (e + ew + (2 * e if add else 0)) + vectors
        # s (or x), dy and ds in, one gradient of the sum (or of x) out; weight in, its gradient out
        bwd = n * (2 * e + ew + (e if add else 0)) + 2 * vectors
        return {"bytes": fwd + (bwd if train else 0), "flops": n * (5 + (10 if train else 0))}
    if op == "swiglu":
        n = case["rows"] * case["cols"]
        return {"bytes": n * e * (3 + (5 if train else 0)), "flops": n * (6 + (14 if train else 0))}
    if op in ("rotary_embedding", "rope", "qk_norm_rope"):
        n = case["batch"] * case["seq"] * (case["q_heads"] + case["kv_heads"]) * case["head_dim"]
        et = 4 if case["tables"] == "fp32" else 2
        width = 2 * case["half"] if op == "rotary_embedding" else 2 * case["head_dim"]
        tables = case["seq"] * width * et
        eo = e if op == "rotary_embedding" else max(e, et)
        norm = op == "qk_norm_rope"
        bwd = n * (eo + e + (e if norm else 0)) + tables
        return {"bytes": n * (e + eo) + tables + (bwd if train else 0), "flops": n * ((3 + (4 if norm else 0)) * (2 if train else 1))}
    tokens = case["batch"] * case["seq"] if op == "attn" else case["total"]
    hq, hkv, d = case["q_heads"], case["kv_heads"], case["head_dim"]
    fwd = tokens * d * e * (2 * hq + 2 * hkv)
    bwd = tokens * d * e * (4 * hq + 4 * hkv)  # q, k, v, o, dO in; dq, dk, dv out
    return {"bytes": fwd + (bwd if train else 0), "flops": 4 * d * hq * _pairs(case) * (3.5 if train else 1.0)}


def tolerance(case: dict) -> dict:
    """Four times the distance from float64 that was measured, which is what the storage type's rounding gives."""
    if case["op"] in ("attn", "attn_varlen"):
        # P and dS enter the products in the inputs' type; the longest sums have 16384 terms
        return {"rel": {"bf16": 1.6e-2, "fp16": 2e-3, "fp32": 2.5e-6}[case["dtype"]]}
    # one to three roundings of an output; fp32 keeps those of a row's sums and of the weight gradients' column sums
    return {"rel": {"bf16": 1.4e-2, "fp16": 1.5e-3, "fp32": 1e-6}[case["dtype"]]}


# ------------------------------------------------------------------ the same outputs from float64 torch


def _attention(q, k, v, do, causal: bool):
    """One sequence: q, do [s, hq, d], k, v [s, hkv, d] -> o and, with a cotangent, dq, dk, dv; one q head at a time."""
    s, hq, d = q.shape
    group, scale = hq // k.shape[1], d ** -0.5
    o = torch.empty_like(q)
    dq, dk, dv = (torch.zeros_like(t) for t in (q, k, v)) if do is not None else (None, None, None)
    rows = max(1, (1 << 28) // max(s, 1))  # query rows at a time: 2 GiB of scores
    for h in range(hq):
        kh, vh = k[:, h // group].contiguous(), v[:, h // group].contiguous()
        kt, vt = kh.t().contiguous(), vh.t().contiguous()
        for r in range(0, s, rows):
            qh = q[r:r + rows, h].contiguous()
            p = qh @ kt
            p *= scale
            if causal:
                at = torch.arange(r, r + qh.shape[0], device=q.device)
                p.masked_fill_(torch.arange(s, device=q.device)[None] > at[:, None], float("-inf"))
            p = torch.softmax(p, dim=-1)
            oh = p @ vh
            o[r:r + rows, h] = oh
            if do is None:
                continue
            gh = do[r:r + rows, h].contiguous()
            dv[:, h // group] += p.t().contiguous() @ gh
            ds = gh @ vt
            ds -= (gh * oh).sum(-1, keepdim=True)
            ds *= p
            ds *= scale
            dq[r:r + rows, h] = ds @ kh
            dk[:, h // group] += ds.t().contiguous() @ qh
    return (o,) if do is None else (o, dq, dk, dv)


def _rms(x):
    return x * torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + EPS)


def _rope(x, cos, sin):
    first, second = x.chunk(2, dim=-1)
    return x * cos[:, None] + torch.cat((-second, first), dim=-1) * sin[:, None]


def _rotary(x, cos, sin, interleaved: bool):
    half = cos.shape[-1]
    c, s = cos[:, None], sin[:, None]
    if interleaved:
        u, v = x[..., 0:2 * half:2], x[..., 1:2 * half:2]
        turned = torch.stack((u * c - v * s, u * s + v * c), dim=-1).flatten(-2)
    else:
        u, v = x[..., :half], x[..., half:2 * half]
        turned = torch.cat((u * c - v * s, u * s + v * c), dim=-1)
    return torch.cat((turned, x[..., 2 * half:]), dim=-1)


def exact(case: dict, seed: int):
    state = prepare(case, seed)
    op, train = case["op"], case["train"]

    def wide(name):
        t = state[name]
        return None if t is None else t.detach().double()

    dy = tuple(t.double() for t in state["dy"])
    if op in ("attn", "attn_varlen"):
        q, k, v = wide("q"), wide("k"), wide("v")
        do = dy[0] if train else None
        if op == "attn":
            parts = [_attention(q[b], k[b], v[b], None if do is None else do[b], case["causal"]) for b in range(case["batch"])]
            return tuple(torch.stack(ts) for ts in zip(*parts))
        cuts = state["cu_seqlens"].tolist()
        parts = [_attention(q[i:j], k[i:j], v[i:j], None if do is None else do[i:j], case["causal"])
                 for i, j in zip(cuts, cuts[1:])]
        return tuple(torch.cat(ts) for ts in zip(*parts))
    names = {"rms_norm": ("x", "weight", "bias"), "add_rms_norm": ("x", "residual", "weight"), "swiglu": ("a", "b"),
             "rotary_embedding": ("q", "k"), "rope": ("q", "k"), "qk_norm_rope": ("q", "k", "q_weight", "k_weight")}[op]
    inputs = [wide(n) for n in names]
    held = [t.requires_grad_(train) for t in inputs if t is not None]
    with torch.set_grad_enabled(train):
        if op == "rms_norm":
            y = _rms(inputs[0]) * inputs[1]
            out = (y if inputs[2] is None else y + inputs[2],)
        elif op == "add_rms_norm":
            s = inputs[0] + inputs[1]
            out = (_rms(s) * (inputs[2] + case["offset"]), s)
        elif op == "swiglu":
            out = (torch.nn.functional.silu(inputs[0]) * inputs[1],)
        elif op == "rotary_embedding":
            out = tuple(_rotary(t, wide("cos"), wide("sin"), case["interleaved"]) for t in inputs)
        elif op == "rope":
            out = tuple(_rope(t, wide("cos"), wide("sin")) for t in inputs)
        else:
            q, k, qw, kw = inputs
            out = tuple(_rope(_rms(t) * w, wide("cos"), wide("sin")) for t, w in ((q, qw), (k, kw)))
        grads = torch.autograd.grad(out, held, dy) if train else ()
    return tuple(t.detach() for t in out) + tuple(grads)
