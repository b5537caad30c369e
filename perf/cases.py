"""What this library is timed on: the attention block and the projections of a decoder, through the public entry points.

A case is a dict of plain values.  Its "kind" says which part of a decoder's work it is:

* ``step``    one token per sequence at a time through `layers` layers' in-place caches: append + attention, `tokens` times over
* ``ragged``  the same for sequences of different lengths with caches of their own
* ``chunk``   several tokens per sequence at once: a prompt, a chunk of one, or a few proposed tokens to verify
* ``project`` Q4_0 weights times activation rows, `layers` matrices one after the other
* ``kivi``    a session over the u8 stores with affine parameters: a prompt, then `tokens` single tokens

A pass starts from the same lengths every time: the caches are truncated to `past` tokens first (what a host does
with tokens it rejected), a session is reset.  Several layers stand behind one pass so that a launch does not find its
cache in the Infinity Cache, as in a decoder.
"""
import math

import numpy as np
import torch

import tract_amd as ta

_NP = {"f16": np.float16, "f32": np.float32}
_TORCH = {"f16": torch.float16, "f32": torch.float32}
_STORE = {"plain": None, "q8_0": ta.Q8_0, "q4_0": ta.Q4_0}


def _step(name, dtype, store, batch, heads, kv_heads, dim, past, tokens, layers, rope):
    return {"name": name, "kind": "step", "dtype": dtype, "store": store, "batch": batch, "heads": heads, "kv_heads": kv_heads,
            "dim": dim, "past": past, "tokens": tokens, "layers": layers, "rope": rope}


def _chunk(name, dtype, store, batch, heads, kv_heads, dim, past, chunk, layers):
    return {"name": name, "kind": "chunk", "dtype": dtype, "store": store, "batch": batch, "heads": heads, "kv_heads": kv_heads,
            "dim": dim, "past": past, "chunk": chunk, "layers": layers}


def _project(name, dtype, rows, n, k, layers):
    return {"name": name, "kind": "project", "dtype": dtype, "rows": rows, "n": n, "k": k, "layers": layers}


def listed():
    return [
        # a small f32 model with one kv head per query head, early in a conversation: launches and host calls are all there is
        _step("step_f32_short", "f32", "plain", 1, 32, 32, 64, 200, 4, 4, False),
        # one user of a grouped-head decoder at a long context, with the rotary embedding its graph has around the cache
        _step("step_f16_one_user", "f16", "plain", 1, 32, 8, 128, 8192, 4, 4, True),
        # the serving batch: 8 users, 8192 tokens each
        _step("step_f16_batch", "f16", "plain", 8, 32, 8, 128, 8192, 4, 4, False),
        # the same users over caches quantised to a quarter, at a length that is no multiple of anything
        _step("step_q4_0_batch", "f16", "q4_0", 8, 32, 8, 128, 4501, 4, 4, False),
        # a continuous batch: 64 sequences of 512 to 32768 tokens
        {"name": "ragged_f16", "kind": "ragged", "dtype": "f16", "store": "plain", "seqs": 64, "shortest": 512, "longest": 32768,
         "heads": 32, "kv_heads": 8, "dim": 128, "tokens": 4},
        # the last of eight 512-token chunks of a 4096-token prompt
        _chunk("chunk_f16", "f16", "plain", 1, 32, 8, 128, 3584, 512, 4),
        # a few proposed tokens per user to verify, over a long context
        _chunk("verify_f16", "f16", "plain", 4, 32, 8, 128, 5000, 6, 4),
        # a prompt through an f32 model
        _chunk("prompt_f32", "f32", "plain", 1, 32, 8, 128, 0, 1000, 1),
        # the widest projection of a decoder for one token
        _project("project_f16_token", "f16", 1, 14336, 4096, 4),
        # the projection back for a chunk of a prompt
        _project("project_f16_chunk", "f16", 512, 4096, 14336, 4),
        # a short prompt through a square projection of an f32 model
        _project("project_f32_prompt", "f32", 150, 4096, 4096, 4),
        # a session over the affine u8 stores: a prompt, then an answer
        {"name": "kivi_session", "kind": "kivi", "dtype": "f16", "batch": 2, "heads": 32, "kv_heads": 8, "dim": 128, "prompt": 1500,
         "tokens": 16},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "ragged", "chunk", "chunk", "chunk", "project", "project", "project", "kivi"])
    heads, kv_heads = rng.choice([(32, 8), (32, 8), (32, 32), (64, 8), (40, 8), (14, 2)])
    dim = rng.choice([128, 128, 64])
    if kind == "step":
        store = rng.choice(["plain", "plain", "q8_0", "q4_0"])
        dtype = rng.choice(["f16", "f16", "f32"]) if store == "plain" else "f16"
        dim = dim if store == "plain" else 128
        batch = _log(rng, 1, 32)
        past = _log(rng, 100, 20000)
        past = max(100, min(past, 131072 // batch * 8 // kv_heads))
        return _unnamed(_step("", dtype, store, batch, heads, kv_heads, dim, past, 4, rng.choice([2, 4]), rng.random() < 0.5))
    if kind == "ragged":
        if kv_heads == 32:
            heads, kv_heads = 32, 8
        longest = _log(rng, 1000, 32768)
        store = rng.choice(["plain", "plain", "q8_0", "q4_0"])
        return {"kind": kind, "dtype": "f16", "store": store, "seqs": _log(rng, 3, 64), "shortest": max(1, longest // rng.choice([3, 20, 64])),
                "longest": longest, "heads": heads, "kv_heads": kv_heads, "dim": 128 if store != "plain" else dim, "tokens": 4}
    if kind == "chunk":
        dtype = rng.choice(["f16", "f16", "f32"])
        store = rng.choice(["plain", "plain", "q8_0", "q4_0"]) if dtype == "f16" and dim == 128 else "plain"
        if rng.random() < 0.4:     # a few tokens to verify
            batch, chunk, past = _log(rng, 1, 8), rng.randint(2, 16), _log(rng, 200, 8192)
            layers = 4
        else:                      # a prompt or a chunk of one
            batch, chunk, past = rng.choice([1, 1, 2, 3]), _log(rng, 32, 2048), rng.choice([0, 0, _log(rng, 100, 4096)])
            layers = 2
        if dtype == "f32" or store != "plain":
            layers = 1
            batch = max(1, min(batch, (1 << 25) // (heads * chunk * (past + chunk))))
            past = min(past, max(0, (1 << 25) // (heads * chunk * batch) - chunk))
            chunk = min(chunk, 1000)
        return _unnamed(_chunk("", dtype, store, batch, heads, kv_heads, dim, past, chunk, layers))
    if kind == "project":
        n, k = rng.choice([(4096, 4096), (1024, 4096), (14336, 4096), (4096, 14336), (2816, 1024), (1000, 2080)])
        dtype = rng.choice(["f16", "f16", "f32"])
        rows = rng.choice([rng.randint(1, 16), _log(rng, 1, 1024)])
        if dtype == "f32":
            rows = min(rows, 512)
        return _unnamed(_project("", dtype, rows, n, k, 4))
    batch = rng.choice([1, 2, 3, 4])
    if kv_heads == 32:
        heads, kv_heads = 32, 8
    return {"kind": kind, "dtype": "f16", "batch": batch, "heads": heads, "kv_heads": kv_heads, "dim": 128, "prompt": _log(rng, 64, 3000 // batch),
            "tokens": rng.choice([4, 16])}


def _unnamed(case):
    del case["name"]
    return case


# ---- inputs ------------------------------------------------------------------------------------------------


class _Memory:
    """Device memory of a cache's planes as torch sees it (what a step appended is read back through this); the tensor
    made of it keeps this object alive, and this object the cache."""

    def __init__(self, cache, ptr, shape, strides, dtype):
        self.cache = cache
        size = np.dtype(dtype).itemsize
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "strides": tuple(s * size for s in strides),
                                         "typestr": np.dtype(dtype).str, "version": 2}


def _wrap(t):
    """A torch tensor as the library's DeviceTensor over the same memory."""
    return ta.DeviceTensor(t.shape, np.dtype(str(t.dtype).replace("torch.", "")), ptr=t.data_ptr(), owner=t)


class _Inputs:
    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(int(seed))
        self.rng = np.random.default_rng(int(seed))

    def normal(self, shape, dtype, scale=1.0, outliers=False):
        t = torch.randn(tuple(shape), generator=self.gen, device="cuda", dtype=torch.float32) * scale
        if outliers:   # about 1 % of the channels are 20 times as large, as keys have them
            t[..., :: 96] *= 20.0
        return t.to(_TORCH[dtype])


def _caches(case, x, store, batch, past, extra, layers):
    """`layers` states whose caches hold `past` tokens and have room for `extra` more."""
    dt, hkv, d = case["dtype"], case["kv_heads"], case["dim"]
    states = []
    for _ in range(layers):
        st = ta.InPlaceKvSdpa(axis=2, causal=True, storage_format=store).state()
        for c in (st.k, st.v):
            c.reserve(past + extra, like=((batch, hkv, 1, d), _NP[dt]))
            if past:
                rows = x.normal((batch, hkv, past, d), dt, outliers=store is not None)
                torch.cuda.synchronize()
                c.push(_wrap(rows))
                ta.synchronize()
        states.append(st)
    return states


def _appended(cache, batch, heads, dim, past, n, dtype):
    """The n rows after `past` of a plain cache's planes."""
    ptr, _, pitch = cache.raw()
    whole = torch.as_tensor(_Memory(cache, ptr, (batch, heads, past + n, dim), (heads * pitch * dim, pitch * dim, dim, 1), _NP[dtype]), device="cuda")
    return whole[:, :, past:]


def _rotary(x, positions, dim, dtype):
    """cos and sin rows [len(positions), dim] as an exported decoder makes them."""
    inv = 10000.0 ** (-torch.arange(0, dim, 2, device="cuda", dtype=torch.float32) / dim)
    angle = torch.tensor(positions, device="cuda", dtype=torch.float32)[:, None] * inv[None, :]
    angle = torch.cat([angle, angle], dim=1)
    return angle.cos().to(_TORCH[dtype]), angle.sin().to(_TORCH[dtype])


def _prepare_step(case, x):
    b, hq, hkv, d, dt = case["batch"], case["heads"], case["kv_heads"], case["dim"], case["dtype"]
    past, n = case["past"], case["tokens"]
    states = _caches(case, x, _STORE[case["store"]], b, past, n, case["layers"])
    calls, outs, keep = [], [], []
    for t in range(n):
        cos, sin = _rotary(x, [past + t], d, dt)
        cs = [_wrap(r.reshape(1, 1, 1, d)) for r in (cos, sin)] if case["rope"] else []
        for st in states:
            q, k, v = x.normal((b, hq, 1, d), dt), x.normal((b, hkv, 1, d), dt), x.normal((b, hkv, 1, d), dt)
            out = torch.empty_like(q)
            outs.append(out)
            keep += [q, k, v]
            calls.append((st, [_wrap(q), _wrap(k), _wrap(v)] + cs, _wrap(out)))
    if case["store"] == "plain":
        outs += [_appended(c, b, hkv, d, past, n, dt) for st in states for c in (st.k, st.v)]
    return {"past": past, "caches": [c for st in states for c in (st.k, st.v)], "calls": calls, "outs": outs, "rope": case["rope"], "keep": keep}


def _run_step(s):
    for c in s["caches"]:
        c.truncate(s["past"])
    if s["rope"]:
        for st, args, out in s["calls"]:
            st.eval_rope_into(*args, out)
    else:
        for st, args, out in s["calls"]:
            st.eval_into(*args, out)
    return s["outs"]


def _lengths(case, rng):
    return [int(n) for n in rng.integers(case["shortest"], case["longest"], size=case["seqs"], endpoint=True)]


def _prepare_ragged(case, x):
    n, hq, hkv, d, dt = case["seqs"], case["heads"], case["kv_heads"], case["dim"], case["dtype"]
    lens = _lengths(case, np.random.default_rng(7))   # the lengths are the case's, not the seed's
    ks, vs = [], []
    for length in lens:
        for many in (ks, vs):
            c = ta.InPlaceKvCache(2, _STORE[case["store"]])
            c.reserve(length + case["tokens"], like=((1, hkv, 1, d), _NP[dt]))
            rows = x.normal((1, hkv, length, d), dt, outliers=case["store"] != "plain")
            torch.cuda.synchronize()
            c.push(_wrap(rows))
            ta.synchronize()
            many.append(c)
    calls, outs = [], []
    for _ in range(case["tokens"]):
        q, k, v = x.normal((n, hq, 1, d), dt), x.normal((n, hkv, 1, d), dt), x.normal((n, hkv, 1, d), dt)
        out = torch.empty_like(q)
        outs.append(out)
        calls.append((_wrap(q), _wrap(k), _wrap(v), _wrap(out)))
    return {"lens": lens, "ks": ks, "vs": vs, "calls": calls, "outs": outs, "ws": ta.Workspace(n, hq, 1, d)}


def _run_ragged(s):
    for length, k, v in zip(s["lens"], s["ks"], s["vs"]):
        k.truncate(length)
        v.truncate(length)
    for q, k, v, out in s["calls"]:
        ta.inplace_kv_sdpa_eval_ragged(q, k, v, s["ks"], s["vs"], workspace=s["ws"], out=out)
    return s["outs"]


def _prepare_chunk(case, x):
    b, hq, hkv, d, dt, n = case["batch"], case["heads"], case["kv_heads"], case["dim"], case["dtype"], case["chunk"]
    states = _caches(case, x, _STORE[case["store"]], b, case["past"], n, case["layers"])
    calls, outs = [], []
    for st in states:
        q, k, v = x.normal((b, hq, n, d), dt), x.normal((b, hkv, n, d), dt), x.normal((b, hkv, n, d), dt)
        out = torch.empty_like(q)
        outs.append(out)
        calls.append((st, [_wrap(q), _wrap(k), _wrap(v)], _wrap(out)))
    if case["store"] == "plain":
        outs += [_appended(c, b, hkv, d, case["past"], n, dt) for st in states for c in (st.k, st.v)]
    return {"past": case["past"], "caches": [c for st in states for c in (st.k, st.v)], "calls": calls, "outs": outs, "rope": False}


def _q4_0_blocks(w):
    """Canonical Q4_0 blocks of a [n, k] f32 tensor (18 bytes per 32 features: f16 scale, 16 bytes of code pairs)."""
    g = w.reshape(-1, 32)
    at = g.abs().argmax(dim=1, keepdim=True)
    scale = g.gather(1, at) / -8.0
    inv = torch.where(scale == 0, torch.zeros_like(scale), 1.0 / scale)
    codes = (g * inv + 8.5).clamp(0, 15).to(torch.uint8)
    packed = codes[:, :16] | (codes[:, 16:] << 4)
    return torch.cat([scale.to(torch.float16).view(torch.uint8), packed], dim=1).reshape(-1)


def _prepare_project(case, x):
    m, n, k, dt = case["rows"], case["n"], case["k"], case["dtype"]
    calls, outs = [], []
    for _ in range(case["layers"]):
        blocks = _q4_0_blocks(x.normal((n, k), "f32", scale=0.03))
        torch.cuda.synchronize()
        w = ta.Q40Weights(_wrap(blocks), 1, n, k)
        act = x.normal((1, m, k), dt)
        out = torch.empty((1, m, n), device="cuda", dtype=_TORCH[dt])
        outs.append(out)
        calls.append((w, _wrap(act), _wrap(out)))
    return {"op": ta.GgmlGemm(), "calls": calls, "outs": outs}


def _run_project(s):
    op = s["op"]
    for w, act, out in s["calls"]:
        op.eval(act, w, out=out)
    return s["outs"]


def _prepare_kivi(case, x):
    b, hq, hkv, d, dt = case["batch"], case["heads"], case["kv_heads"], case["dim"], case["dtype"]
    st = ta.QuantizedKvSdpa(axis=2).state()
    calls, outs = [], []
    for n in [case["prompt"]] + [1] * case["tokens"]:
        q, k, v = x.normal((b, hq, n, d), dt), x.normal((b, hkv, n, d), dt, outliers=True), x.normal((b, hkv, n, d), dt)
        out = torch.empty_like(q)
        outs.append(out)
        calls.append(([_wrap(q), _wrap(k), _wrap(v)], _wrap(out)))
    return {"st": st, "calls": calls, "outs": outs}


def _run_kivi(s):
    st = s["st"]
    if st.k is not None:
        st.k.reset()
        st.v.reset()
    for args, out in s["calls"]:
        st.eval(args, out=out)
    return s["outs"]


_PREPARE = {"step": _prepare_step, "ragged": _prepare_ragged, "chunk": _prepare_chunk, "project": _prepare_project, "kivi": _prepare_kivi}
_RUN = {"step": _run_step, "ragged": _run_ragged, "chunk": _run_step, "project": _run_project, "kivi": _run_kivi}


def prepare(case, seed):
    ta.runtime_for_name("rocm")
    state = _PREPARE[case["kind"]](case, _Inputs(seed))
    torch.cuda.synchronize()
    return {"run": _RUN[case["kind"]], "state": state}


def run(state):
    return state["run"](state["state"])


# ---- what a pass cannot do without ---------------------------------------------------------------------------

_ROW = {"f16": lambda d: 2 * d, "f32": lambda d: 4 * d, "q8_0": lambda d: d // 32 * 34, "q4_0": lambda d: d // 32 * 18}


def work(case):
    size = {"f16": 2, "f32": 4}[case["dtype"]]
    kind = case["kind"]
    if kind == "project":
        m, n, k = case["rows"], case["n"], case["k"]
        return {"bytes": case["layers"] * (n * (k // 32) * 18 + m * (n + k) * size), "flops": case["layers"] * 2 * m * n * k}
    hq, hkv, d = case["heads"], case["kv_heads"], case["dim"]
    if kind == "kivi":
        b, p, n = case["batch"], case["prompt"], case["tokens"]
        new = b * (p + n) * d * size * (2 * hq + 2 * hkv)                      # q, k, v in, out
        coded = b * hkv * (2 * d + 8)                                        # a token's codes and the value parameters
        steps = sum(p + t + 1 for t in range(n))
        return {"bytes": new + coded * (p + n) + coded * steps, "flops": 4 * b * hq * d * (p * p + steps)}
    row = _ROW[case["dtype"] if case["store"] == "plain" else case["store"]](d)
    if kind == "ragged":
        lens = _lengths(case, np.random.default_rng(7))
        keys = sum(length + t + 1 for length in lens for t in range(case["tokens"]))
        new, tokens = case["seqs"] * case["tokens"], 1
    elif kind == "step":
        tokens = case["layers"] * case["tokens"]
        keys = case["batch"] * case["layers"] * sum(case["past"] + t + 1 for t in range(case["tokens"]))
        new = case["batch"] * tokens
    else:
        n = case["chunk"]
        new = case["batch"] * case["layers"] * n
        keys = case["batch"] * case["layers"] * (case["past"] + n)             # each key row is read once for its chunk
        pairs = case["batch"] * case["layers"] * (n * case["past"] + n * (n + 1) // 2)
        return {"bytes": keys * hkv * 2 * row + new * d * size * (2 * hq + 2 * hkv), "flops": 4 * pairs * hq * d}
    return {"bytes": keys * hkv * 2 * row + new * d * size * (2 * hq + 2 * hkv), "flops": 4 * keys * hq * d}


def tolerance(case):
    """About four times what a float64 restatement of the case measures: f32 attention and projections 1e-7 .. 4e-7 (largest
    7e-6); f16 2e-4 .. 3.6e-4 (2e-3: results and probabilities are rounded to f16); block-quantised and affine stores up to
    1.5e-3 (0.07), where keys of outlying channels enter the products as f16 and the softmax is sharp."""
    if case["dtype"] == "f32":
        return {"rel": 2e-6}
    if case["kind"] == "kivi" or case.get("store", "plain") != "plain":
        return {"rel": 6e-3, "max": 0.3}
    return {"rel": 1.5e-3, "max": 1e-2}
