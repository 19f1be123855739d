"""The work a program has this library do, as cases that can be timed.

A case is one pass through the public entry points of ``mfattn``: a packed
attention step (block map, forward and, in training, backward), a KV-cached
decode step, the attention prologue, or a segmented short convolution.  Sizes
are those of the benchmark layouts (16 query and 8 key heads of 64, rows of
4096-32768 packed tokens, caches of up to 8192 slots, 1024 convolution
channels) and the smaller and odd ones around them.

``listed()`` names the cases, ``draw(rng)`` gives more of the same ranges,
``prepare`` makes what a program holds before the call, ``run`` is the call.
"""

from __future__ import annotations

import math
import pathlib
import sys

import numpy as np
import torch

_PACKAGE = pathlib.Path(__file__).resolve().parents[1] / "minifield-training_amd"
if str(_PACKAGE) not in sys.path:
    sys.path.insert(0, str(_PACKAGE))

D = 64  # head dimension of every configuration
_DTYPES = {"bfloat16": torch.bfloat16, "float32": torch.float32}
_BYTES = {"bfloat16": 2, "float32": 4}
_EPS, _THETA = 1e-5, 1e6


# --------------------------------------------------------------------------- cases


def _attention(mode, dtype, rows, tokens, heads, kv_heads, spread, low, high, train, layout):
    return {"kind": "attention", "mode": mode, "dtype": dtype, "rows": rows, "tokens": tokens,
            "heads": heads, "kv_heads": kv_heads, "spread": spread, "low": low, "high": high,
            "train": train, "layout": layout}


def _decode(dtype, rows, capacity, heads, kv_heads, low, high, append, layout):
    return {"kind": "decode", "dtype": dtype, "rows": rows, "capacity": capacity, "heads": heads,
            "kv_heads": kv_heads, "low": low, "high": high, "append": append, "layout": layout}


def _prologue(dtype, rows, tokens, heads, kv_heads, train, layout):
    return {"kind": "prologue", "dtype": dtype, "rows": rows, "tokens": tokens, "heads": heads,
            "kv_heads": kv_heads, "spread": "log", "low": 32, "high": 2048, "train": train,
            "layout": layout}


def _conv(mode, dtype, rows, tokens, channels, taps, train, layout):
    return {"kind": "conv", "mode": mode, "dtype": dtype, "rows": rows, "tokens": tokens,
            "channels": channels, "taps": taps, "spread": "log", "low": 32, "high": 2048,
            "train": train, "layout": layout}


def listed():
    return [
        # the smallest training step anyone runs: a unit test, a smoke run, a
        # debugging session in float32; launches and host time are all of it
        {"name": "tiny_fp32_train",
         **_attention("causal", "float32", 2, 256, 4, 2, "uniform", 1, 64, True, 101)},
        # fine-tuning with one packed row per step on one GPU: too few tiles
        # to fill the chip
        {"name": "one_row_train",
         **_attention("causal", "bfloat16", 1, 2048, 16, 8, "geometric", 16, 512, True, 11)},
        # encoder pre-training at the 350M shape: the headline workload
        {"name": "encoder_train",
         **_attention("packed", "bfloat16", 8, 4096, 16, 8, "log", 32, 2048, True, 202)},
        # causal pre-training on packed documents
        {"name": "causal_train",
         **_attention("causal", "bfloat16", 4, 8192, 16, 8, "geometric", 16, 512, True, 303)},
        # one long row of many short samples (chat turns, classification):
        # almost every tile is masked
        {"name": "short_segments_train",
         **_attention("causal", "bfloat16", 1, 32768, 16, 8, "uniform", 16, 128, True, 505)},
        # a float32 reference step at a ragged length, to check a bf16 run against
        {"name": "fp32_train",
         **_attention("causal", "float32", 2, 1499, 16, 8, "geometric", 16, 512, True, 12)},
        # embedding a batch of padded texts, no packing: forward only
        {"name": "padded_encode",
         **_attention("padded", "bfloat16", 24, 333, 16, 8, "uniform", 83, 333, False, 13)},
        # prefill of one long prompt of odd length: forward only, one segment
        {"name": "prompt_prefill",
         **_attention("causal", "bfloat16", 1, 5003, 16, 8, "whole", 5003, 5003, False, 14)},
        # one user's next token, with the cache write: latency
        {"name": "decode_one",
         **_decode("bfloat16", 1, 4096, 16, 8, 2000, 4095, True, 15)},
        # a serving batch's next token over ragged caches: bandwidth
        {"name": "decode_batch",
         **_decode("bfloat16", 64, 8192, 16, 8, 128, 8192, False, 404)},
        # query/key norm and rotary embedding around a packed attention layer
        {"name": "prologue_train", **_prologue("bfloat16", 8, 4096, 16, 8, True, 202)},
        # the encoder's gated short convolution over 1024 channels
        {"name": "conv_train", **_conv("packed", "bfloat16", 8, 4096, 1024, 3, True, 202)},
    ]


def _log_int(rng, low, high):
    return min(high, max(low, int(math.exp(rng.uniform(math.log(low), math.log(high + 1))))))


_HEADS = ((16, 8), (16, 8), (32, 8), (8, 8), (12, 4), (4, 2))


def draw(rng):
    """One more case: the listed kinds at sizes spread over their ranges."""
    kind = rng.choice(("attention",) * 5 + ("decode",) * 3 + ("prologue", "conv"))
    layout = rng.randrange(1 << 30)
    dtype = "float32" if rng.random() < 0.15 else "bfloat16"
    heads, kv_heads = rng.choice(_HEADS)
    train = rng.random() < 0.7
    if kind == "decode":
        rows = _log_int(rng, 1, 64)
        capacity = _log_int(rng, 64, 8192)
        high = capacity - 1 if capacity > 1 else 1
        # rows x capacity x key heads of one listed batch at most
        while rows * capacity * kv_heads * _BYTES[dtype] > 64 * 8192 * 8 * 2:
            rows = max(1, rows // 2)
        return _decode(dtype, rows, capacity, heads, kv_heads, max(1, capacity // 64), high,
                       rng.random() < 0.5, layout)
    if kind == "conv":
        taps = rng.choice((3, 3, 4))
        channels = rng.choice((512, 768, 1024))
        tokens = _log_int(rng, 64, 4096)
        rows = max(1, _log_int(rng, 64, (16384 if dtype == "float32" else 32768)) // tokens)
        return _conv(rng.choice(("packed", "causal")), dtype, rows, tokens, channels, taps, train,
                     layout)
    if kind == "prologue":
        tokens = _log_int(rng, 64, 4096)
        limit = 32768 * 24 // (heads + kv_heads) // (2 if dtype == "float32" else 1)
        rows = max(1, _log_int(rng, 64, limit) // tokens)
        return _prologue(dtype, rows, tokens, heads, kv_heads, train, layout)
    while True:
        mode = rng.choice(("causal", "causal", "packed", "padded"))
        total = _log_int(rng, 64, 4096 if dtype == "float32" else 32768)
        tokens = min(total, _log_int(rng, 48, 1024 if mode == "padded" else 16384))
        rows = max(1, total // tokens)
        if mode == "padded":
            spread, low, high = "uniform", max(1, tokens // 4), tokens
        else:
            spread, low, high = rng.choice((("geometric", 16, 512), ("log", 32, 2048),
                                            ("uniform", 16, 128), ("uniform", 64, 1024),
                                            ("whole", tokens, tokens)))
        case = _attention(mode, dtype, rows, tokens, heads, kv_heads, spread, low, high, train,
                          layout)
        # at most what the largest listed cases cost
        if work(case)["flops"] <= (8e9 if dtype == "float32" else 2e11):
            return case


# --------------------------------------------------------------------------- layouts


def _segments(case):
    """Packed segment ids [rows, tokens] (0: padding) of the case's layout."""
    rng = np.random.default_rng(case["layout"])
    rows, tokens = case["rows"], case["tokens"]
    seg = np.zeros((rows, tokens), dtype=np.int32)
    low, high = case["low"], case["high"]
    for r in range(rows):
        at, ident = 0, 1
        while True:
            if case["spread"] == "whole":
                size = tokens
            elif case["spread"] == "uniform":
                size = int(rng.integers(low, high + 1))
            elif case["spread"] == "log":
                size = int(math.exp(rng.uniform(math.log(low), math.log(high))))
            else:  # geometric of mean `high`, at least `low`
                size = max(low, int(rng.geometric(1.0 / high)))
            if at == 0:
                size = min(size, tokens)  # a row holds at least one (cut) sample
            if at + size > tokens:
                break
            seg[r, at:at + size] = ident
            at, ident = at + size, ident + 1
    return seg


def _lengths(case):
    """Valid lengths of a padded batch or of a batch of caches."""
    rng = np.random.default_rng(case["layout"])
    return rng.integers(case["low"], case["high"] + 1, size=case["rows"]).astype(np.int32)


def _runs(seg):
    """(row, start, stop) of every run of one nonzero id."""
    found = []
    for r, ids in enumerate(seg):
        edges = np.flatnonzero(np.diff(ids)) + 1
        for a, b in zip(np.concatenate(([0], edges)), np.concatenate((edges, [len(ids)]))):
            if ids[a]:
                found.append((r, int(a), int(b)))
    return found


def _positions(seg):
    pos = np.zeros_like(seg)
    for r, a, b in _runs(seg):
        pos[r, a:b] = np.arange(b - a)
    return pos


# --------------------------------------------------------------------------- inputs


def prepare(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    dtype = _DTYPES[case["dtype"]]

    def normal(*shape, scale=1.0):
        return (torch.randn(shape, generator=gen, device=dev) * scale).to(dtype)

    b, h, kvh = case["rows"], case.get("heads"), case.get("kv_heads")
    state = {"case": case}
    if case["kind"] == "attention":
        t = case["tokens"]
        if case["mode"] == "padded":
            mask = np.arange(t)[None, :] < _lengths(case)[:, None]
            state["seg"] = None
        else:
            seg = _segments(case)
            mask = seg != 0
            state["seg"] = torch.from_numpy(seg).to(dev)
        state["mask"] = torch.from_numpy(mask.astype(np.int32)).to(dev)
        # unit-variance heads, as the query/key norm leaves them
        state["q"], state["k"], state["v"] = normal(b, t, h, D), normal(b, t, kvh, D), normal(b, t, kvh, D)
        if case["train"]:
            state["dout"] = normal(b, t, h, D)
            for name in ("q", "k", "v"):
                state[name].requires_grad_()
    elif case["kind"] == "decode":
        cap = case["capacity"]
        lengths = torch.from_numpy(_lengths(case)).to(dev)
        state["q"] = normal(b, 1, h, D)
        state["k_cache"], state["v_cache"] = normal(b, cap, kvh, D), normal(b, cap, kvh, D)
        if case["append"]:
            state["k_new"], state["v_new"] = normal(b, 1, kvh, D), normal(b, 1, kvh, D)
            state["position"] = lengths - 1
        else:
            state["lengths"] = lengths
    elif case["kind"] == "prologue":
        t = case["tokens"]
        state["positions"] = torch.from_numpy(_positions(_segments(case))).to(dev)
        state["q"], state["k"] = normal(b, t, h, D), normal(b, t, kvh, D)
        state["q_gain"] = (1 + 0.1 * torch.randn(D, generator=gen, device=dev)).to(dtype)
        state["k_gain"] = (1 + 0.1 * torch.randn(D, generator=gen, device=dev)).to(dtype)
        if case["train"]:
            state["dq"], state["dk"] = normal(b, t, h, D), normal(b, t, kvh, D)
            for name in ("q", "k", "q_gain", "k_gain"):
                state[name].requires_grad_()
    else:
        t, c = case["tokens"], case["channels"]
        state["seg"] = torch.from_numpy(_segments(case)).to(dev)
        state["b"], state["c"], state["v"] = normal(b, t, c), normal(b, t, c), normal(b, t, c)
        state["taps"] = normal(c, case["taps"], scale=0.5)
        if case["train"]:
            state["dout"] = normal(b, t, c)
            for name in ("b", "c", "v", "taps"):
                state[name].requires_grad_()
    return state


# --------------------------------------------------------------------------- the call


def run(state):
    case = state["case"]
    return {"attention": _run_attention, "decode": _run_decode, "prologue": _run_prologue,
            "conv": _run_conv}[case["kind"]](case, state)


def _run_attention(case, s):
    from mfattn import _lib, ops
    from mfattn.kernels import attention, bidirectional

    t = case["tokens"]
    mode = {"causal": _lib.MODE_PACKED_CAUSAL, "packed": _lib.MODE_PACKED_BIDIR,
            "padded": _lib.MODE_KEYMASK_BIDIR}[case["mode"]]
    # every batch brings its own layout: its block map is part of the step
    plan = ops.block_map(s["seg"], s["mask"], mode, t, t)
    if case["mode"] == "causal":
        out = attention.packed_causal_attention(s["q"], s["k"], s["v"], s["mask"], s["seg"],
                                                backend="hip", plan=plan)
    else:
        out = bidirectional.attention(s["q"], s["k"], s["v"], s["mask"], s["seg"], plan=plan)
    if not case["train"]:
        return {"out": out}
    dq, dk, dv = torch.autograd.grad(out, (s["q"], s["k"], s["v"]), s["dout"])
    return {"out": out.detach(), "dq": dq, "dk": dk, "dv": dv}


def _run_decode(case, s):
    from mfattn.kernels import attention

    if not case["append"]:
        return {"out": attention.cached_attention(s["q"], s["k_cache"], s["v_cache"], s["lengths"],
                                                  backend="hip")}
    out, k, v = attention.cached_attention_step(s["q"], s["k_new"], s["v_new"], s["k_cache"],
                                                s["v_cache"], s["position"], backend="hip")
    return {"out": out, "k_cache": k, "v_cache": v}


def _run_prologue(case, s):
    from mfattn.kernels import prologue

    q, k = prologue.qk_norm_rope(s["q"], s["k"], s["q_gain"], s["k_gain"], s["positions"], eps=_EPS,
                                 rope_theta=_THETA)
    if not case["train"]:
        return {"q": q, "k": k}
    grads = torch.autograd.grad((q, k), (s["q"], s["k"], s["q_gain"], s["k_gain"]),
                                (s["dq"], s["dk"]))
    return {"q": q.detach(), "k": k.detach(),
            **dict(zip(("dq", "dk", "dq_gain", "dk_gain"), grads))}


def _run_conv(case, s):
    from mfattn.kernels import convolution

    if case["mode"] == "causal":
        out = convolution.gated_depthwise_convolution_segmented(
            s["b"], s["c"], s["v"], s["taps"], s["seg"], kernel_size=case["taps"])
    else:
        out = convolution.gated_centered_convolution(s["b"], s["c"], s["v"], s["taps"], s["seg"])
    if not case["train"]:
        return {"out": out}
    grads = torch.autograd.grad(out, (s["b"], s["c"], s["v"], s["taps"]), s["dout"])
    return {"out": out.detach(), **dict(zip(("db", "dc", "dv", "dtaps"), grads))}


# --------------------------------------------------------------------------- work, tolerance


def _pairs(case):
    """Useful (query, key) pairs per head."""
    if case["mode"] == "padded":
        return int(case["tokens"] * _lengths(case).astype(np.int64).sum())
    total = 0
    for _, a, b in _runs(_segments(case)):
        n = b - a
        total += n * (n + 1) // 2 if case["mode"] == "causal" else n * n
    return total


def work(case):
    size = _BYTES[case["dtype"]]
    if case["kind"] == "attention":
        tokens, h, kvh = case["rows"] * case["tokens"], case["heads"], case["kv_heads"]
        rows = 2 * h + 2 * kvh  # q, k, v, out
        if case["train"]:
            rows += 2 * h + 2 * kvh  # dout, dq, dk, dv
        # scores and P V; in training also dP, dV, dK, dQ
        flops = (12 if case["train"] else 4) * D * h * _pairs(case)
        return {"bytes": tokens * (rows * D * size + 8), "flops": flops}
    if case["kind"] == "decode":
        total = int(_lengths(case).astype(np.int64).sum())
        h, kvh = case["heads"], case["kv_heads"]
        nbytes = 2 * total * kvh * D * size + 2 * case["rows"] * h * D * size + 4 * case["rows"]
        if case["append"]:
            nbytes += 2 * case["rows"] * kvh * D * size
        return {"bytes": nbytes, "flops": 4 * D * h * total}
    if case["kind"] == "prologue":
        values = case["rows"] * case["tokens"] * (case["heads"] + case["kv_heads"]) * D
        # forward: read and write; backward: read the gradients, write the inputs'
        return {"bytes": values * size * (4 if case["train"] else 2) + 4 * case["rows"] * case["tokens"],
                "flops": values * (22 if case["train"] else 8)}
    values = case["rows"] * case["tokens"] * case["channels"]
    # b, c, v -> out; backward: dout -> db, dc, dv
    return {"bytes": values * size * (8 if case["train"] else 4) + 4 * case["rows"] * case["tokens"],
            "flops": values * case["taps"] * (8 if case["train"] else 2)}


def tolerance(case):
    # measured as the relative 2-norm error against 64 bits and stated about
    # four times as large: float32 sums are up to 7e-7 off, and bf16 results
    # carry their own rounding (2e-3) and that of the probabilities, of the
    # normalised values or of the taps' sums (up to 3.6e-3 in all)
    if case["dtype"] == "float32":
        return {"rel": 4e-6}
    return {"rel": 1e-2}


# --------------------------------------------------------------------------- 64 bits


def exact(case, seed):
    s = {n: x.detach().double() if isinstance(x, torch.Tensor) and x.is_floating_point() else x
         for n, x in prepare(case, seed).items()}
    return {"attention": _exact_attention, "decode": _exact_decode, "prologue": _exact_prologue,
            "conv": _exact_conv}[case["kind"]](case, s)


def _exact_attention(case, s):
    q, k, v, train = s["q"], s["k"], s["v"], case["train"]
    group, scale = case["heads"] // case["kv_heads"], D ** -0.5
    res = {"out": torch.zeros_like(q)}
    if train:
        res.update(dq=torch.zeros_like(q), dk=torch.zeros_like(k), dv=torch.zeros_like(v))
    if case["mode"] == "padded":
        jobs = [(r, slice(0, case["tokens"]), slice(0, int(n))) for r, n in enumerate(_lengths(case))]
    else:
        jobs = [(r, slice(a, b), slice(a, b)) for r, a, b in _runs(_segments(case))]
    for r, qs, ks in jobs:
        # a few key heads at a time, so that the scores fit
        n = (qs.stop - qs.start) * (ks.stop - ks.start) * group
        step = max(1, min(case["kv_heads"], (1 << 27) // max(n, 1)))
        for h0 in range(0, case["kv_heads"], step):
            kh = slice(h0, min(h0 + step, case["kv_heads"]))
            qh = slice(kh.start * group, kh.stop * group)
            x = q[r, qs, qh].transpose(0, 1)
            y = k[r, ks, kh].transpose(0, 1).repeat_interleave(group, 0)
            z = v[r, ks, kh].transpose(0, 1).repeat_interleave(group, 0)
            p = torch.matmul(x, y.transpose(1, 2)) * scale
            if case["mode"] == "causal":
                p.masked_fill_(torch.ones(p.shape[1:], dtype=torch.bool, device=p.device).triu(1),
                               -math.inf)
            p = p.softmax(-1)
            o = torch.matmul(p, z)
            res["out"][r, qs, qh] = o.transpose(0, 1)
            if train:
                g = s["dout"][r, qs, qh].transpose(0, 1)

                def heads_summed(w):
                    return w.unflatten(0, (-1, group)).sum(1).transpose(0, 1)

                res["dv"][r, ks, kh] = heads_summed(torch.matmul(p.transpose(1, 2), g))
                ds = torch.matmul(g, z.transpose(1, 2))
                ds -= (g * o).sum(-1, keepdim=True)
                ds *= p
                ds *= scale
                res["dq"][r, qs, qh] = torch.matmul(ds, y).transpose(0, 1)
                res["dk"][r, ks, kh] = heads_summed(torch.matmul(ds.transpose(1, 2), x))
    return res


def _exact_decode(case, s):
    group, outs = case["heads"] // case["kv_heads"], []
    for r, n in enumerate(_lengths(case).tolist()):
        k, v = s["k_cache"][r, :n].clone(), s["v_cache"][r, :n].clone()
        if case["append"]:
            k[n - 1], v[n - 1] = s["k_new"][r, 0], s["v_new"][r, 0]
        k = k.transpose(0, 1).repeat_interleave(group, 0)
        v = v.transpose(0, 1).repeat_interleave(group, 0)
        p = (torch.matmul(k, s["q"][r, 0][:, :, None])[..., 0] * D ** -0.5).softmax(-1)
        outs.append(torch.matmul(p[:, None, :], v)[:, 0])
    res = {"out": torch.stack(outs)[:, None]}
    if case["append"]:
        res.update(k_cache=None, v_cache=None)
    return res


def _exact_prologue(case, s):
    # angles in single precision, as rotary embeddings are defined here
    freq = torch.tensor([_THETA ** (-2.0 * i / D) for i in range(D // 2)], dtype=torch.float32)
    angle = (s["positions"].float()[..., None] * freq.to(s["q"].device)).double()
    cos, sin = (torch.cat((f(angle),) * 2, -1)[:, :, None] for f in (torch.cos, torch.sin))

    def forward(x, w):
        n = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + _EPS) * w
        return n * cos + torch.cat((-n[..., D // 2:], n[..., :D // 2]), -1) * sin

    def backward(x, w, g):
        inv = torch.rsqrt((x * x).mean(-1, keepdim=True) + _EPS)
        y, gs = x * inv, g * sin
        dn = g * cos + torch.cat((gs[..., D // 2:], -gs[..., :D // 2]), -1)
        dy = dn * w
        return inv * (dy - y * (dy * y).mean(-1, keepdim=True)), (dn * y).sum((0, 1, 2))

    res = {"q": forward(s["q"], s["q_gain"]), "k": forward(s["k"], s["k_gain"])}
    if case["train"]:
        res["dq"], res["dq_gain"] = backward(s["q"], s["q_gain"], s["dq"])
        res["dk"], res["dk_gain"] = backward(s["k"], s["k_gain"], s["dk"])
    return res


def _exact_conv(case, s):
    taps, seg, t = case["taps"], s["seg"], case["tokens"]
    first = -(taps // 2) if case["mode"] == "packed" else -(taps - 1)
    u, w = s["b"] * s["v"], s["taps"]

    def shifted(x, by):
        """x[t + by], zero outside the row or the token's segment."""
        res = torch.zeros_like(x)
        a, b = max(0, -by), min(t, t - by)
        if a < b:
            same = (seg[:, a:b] == seg[:, a + by:b + by]) & (seg[:, a:b] != 0)
            res[:, a:b] = x[:, a + by:b + by] * same[..., None]
        return res

    mixed = sum(shifted(u, first + i) * w[:, i] for i in range(taps))
    res = {"out": s["c"] * mixed}
    if case["train"]:
        h = s["dout"] * s["c"]
        du = sum(shifted(h, -(first + i)) * w[:, i] for i in range(taps))
        res.update(db=du * s["v"], dc=s["dout"] * mixed, dv=du * s["b"],
                   dtaps=torch.stack([(h * shifted(u, first + i)).sum((0, 1)) for i in range(taps)], 1))
    return res
