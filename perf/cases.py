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
            longest = math.isqrt((1 << 25) // heads)
            if chunk > longest:
                chunk = rng.randint(longest // 2, longest)
            batch = max(1, min(batch, (1 << 25) // (heads * chunk * (past + chunk))))
            past = min(past, max(0, (1 << 25) // (heads * chunk * batch) - chunk))
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


def _past_rows(case, x):
    """The rows that a layer's key or value cache holds before the pass (None for none)."""
    if case["past"]:
        return x.normal((case["batch"], case["kv_heads"], case["past"], case["dim"]), case["dtype"], outliers=case["store"] != "plain")


def _new_rows(case, x, batch, n, outliers=False):
    """q, k and v of n tokens of each of `batch` sequences."""
    hq, hkv, d, dt = case["heads"], case["kv_heads"], case["dim"], case["dtype"]
    return x.normal((batch, hq, n, d), dt), x.normal((batch, hkv, n, d), dt, outliers=outliers), x.normal((batch, hkv, n, d), dt)


def _caches(case, x, extra):
    """A state per layer whose caches hold `past` tokens and have room for `extra` more."""
    dt, hkv, d, past, batch = case["dtype"], case["kv_heads"], case["dim"], case["past"], case["batch"]
    states = []
    for _ in range(case["layers"]):
        st = ta.InPlaceKvSdpa(axis=2, causal=True, storage_format=_STORE[case["store"]]).state()
        for c in (st.k, st.v):
            c.reserve(past + extra, like=((batch, hkv, 1, d), _NP[dt]))
            rows = _past_rows(case, x)
            if rows is not None:
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
    b, hkv, d, dt = case["batch"], case["kv_heads"], case["dim"], case["dtype"]
    past, n = case["past"], case["tokens"]
    states = _caches(case, x, n)
    calls, outs, keep = [], [], []
    for t in range(n):
        cos, sin = _rotary(x, [past + t], d, dt)
        cs = [_wrap(r.reshape(1, 1, 1, d)) for r in (cos, sin)] if case["rope"] else []
        for st in states:
            q, k, v = _new_rows(case, x, b, 1)
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


def _ragged_rows(case, x, lens):
    """Keys, then values, of each sequence in turn."""
    for length in lens:
        for _ in range(2):
            yield x.normal((1, case["kv_heads"], length, case["dim"]), case["dtype"], outliers=case["store"] != "plain")


def _prepare_ragged(case, x):
    n, hq, hkv, d, dt = case["seqs"], case["heads"], case["kv_heads"], case["dim"], case["dtype"]
    lens = _lengths(case, np.random.default_rng(7))   # the lengths are the case's, not the seed's
    rows_of = _ragged_rows(case, x, lens)
    ks, vs = [], []
    for length in lens:
        for many in (ks, vs):
            c = ta.InPlaceKvCache(2, _STORE[case["store"]])
            c.reserve(length + case["tokens"], like=((1, hkv, 1, d), _NP[dt]))
            rows = next(rows_of)
            torch.cuda.synchronize()
            c.push(_wrap(rows))
            ta.synchronize()
            many.append(c)
    calls, outs = [], []
    for _ in range(case["tokens"]):
        q, k, v = _new_rows(case, x, n, 1)
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
    b, hkv, d, dt, n = case["batch"], case["kv_heads"], case["dim"], case["dtype"], case["chunk"]
    states = _caches(case, x, n)
    calls, outs = [], []
    for st in states:
        q, k, v = _new_rows(case, x, b, n)
        out = torch.empty_like(q)
        outs.append(out)
        calls.append((st, [_wrap(q), _wrap(k), _wrap(v)], _wrap(out)))
    if case["store"] == "plain":
        outs += [_appended(c, b, hkv, d, case["past"], n, dt) for st in states for c in (st.k, st.v)]
    return {"past": case["past"], "caches": [c for st in states for c in (st.k, st.v)], "calls": calls, "outs": outs, "rope": False}


def _q4_0_codes(w):
    """Scales (f32, one per 32 elements) and codes of a tensor's Q4_0 blocks."""
    g = w.reshape(-1, 32)
    at = g.abs().argmax(dim=1, keepdim=True)
    scale = g.gather(1, at) / -8.0
    inv = torch.where(scale == 0, torch.zeros_like(scale), 1.0 / scale)
    return scale, (g * inv + 8.5).clamp(0, 15).to(torch.uint8)


def _q4_0_blocks(w):
    """Canonical Q4_0 blocks of a [n, k] f32 tensor (18 bytes per 32 features: f16 scale, 16 bytes of code pairs)."""
    scale, codes = _q4_0_codes(w)
    packed = codes[:, :16] | (codes[:, 16:] << 4)
    return torch.cat([scale.to(torch.float16).view(torch.uint8), packed], dim=1).reshape(-1)


def _project_inputs(case, x):
    """Each layer's weights [n, k] and activation rows."""
    for _ in range(case["layers"]):
        yield x.normal((case["n"], case["k"]), "f32", scale=0.03), x.normal((1, case["rows"], case["k"]), case["dtype"])


def _prepare_project(case, x):
    m, n, k, dt = case["rows"], case["n"], case["k"], case["dtype"]
    calls, outs = [], []
    for weights, act in _project_inputs(case, x):
        blocks = _q4_0_blocks(weights)
        torch.cuda.synchronize()
        w = ta.Q40Weights(_wrap(blocks), 1, n, k)
        out = torch.empty((1, m, n), device="cuda", dtype=_TORCH[dt])
        outs.append(out)
        calls.append((w, _wrap(act), _wrap(out)))
    return {"op": ta.GgmlGemm(), "calls": calls, "outs": outs}


def _run_project(s):
    op = s["op"]
    for w, act, out in s["calls"]:
        op.eval(act, w, out=out)
    return s["outs"]


def _kivi_inputs(case, x):
    """q, k and v of the prompt, then of each single token."""
    return [_new_rows(case, x, case["batch"], n, outliers=True) for n in [case["prompt"]] + [1] * case["tokens"]]


def _prepare_kivi(case, x):
    st = ta.QuantizedKvSdpa(axis=2).state()
    calls, outs = [], []
    for q, k, v in _kivi_inputs(case, x):
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


# ---- the same in 64 bits -----------------------------------------------------------------------------------


def _round_half_away(t):
    return torch.trunc(t.double() + torch.copysign(torch.full_like(t.double(), 0.5), t.double()))


def _stored(rows, store):
    """What a cache of this format holds for these rows, in f64."""
    if store == "plain":
        return rows.double()
    w = rows.float()
    if store == "q4_0":
        scale, codes = _q4_0_codes(w)
        codes = codes.double() - 8.0
    else:
        g = w.reshape(-1, 32)
        scale = g.gather(1, g.abs().argmax(dim=1, keepdim=True)) / 127.0
        inv = torch.where(scale == 0, torch.zeros_like(scale), 1.0 / scale)
        codes = _round_half_away(g * inv).clamp(-128, 127)
    return (codes * scale.to(torch.float16).double()).reshape(rows.shape)


def _attend(q, k, v, causal):
    """Attention of q [hq, n, d] over k and v [hkv, t, d], all f64; causal: the last row of q is the last token."""
    hq, n, d = q.shape
    hkv, t, _ = k.shape
    kt, out = k.transpose(1, 2).contiguous(), torch.empty_like(q)
    step = max(1, (1 << 27) // (hq * t))
    for i in range(0, n, step):
        rows = q[:, i : i + step]
        m = rows.shape[1]
        s = torch.matmul(rows.reshape(hkv, -1, d), kt) / math.sqrt(d)
        if causal:
            sees = torch.arange(t, device="cuda")[None, :] <= (t - n) + torch.arange(i, i + m, device="cuda")[:, None]
            s.view(hkv, -1, m, t).masked_fill_(~sees, -math.inf)
        out[:, i : i + step] = torch.matmul(torch.softmax(s, dim=-1), v).reshape(hq, m, d)
    return out


def _rotate(t, cos, sin):
    half = t.shape[-1] // 2
    return t * cos.double() + torch.cat([-t[..., half:], t[..., :half]], dim=-1) * sin.double()


def _exact_cached(case, x):
    """Steps and chunks: a pass of single tokens over a layer is one causal pass of all of them."""
    b, store, n = case["batch"], case["store"], case["layers"]
    past = [[_past_rows(case, x) for _ in range(2)] for _ in range(n)]
    single = case["kind"] == "step"
    tokens = case["tokens"] if single else 1
    new = [[_new_rows(case, x, b, 1 if single else case["chunk"]) for _ in range(n)] for _ in range(tokens)]   # [token][layer]
    outs, kept = [[None] * n for _ in range(tokens)], []
    for layer in range(n):
        q, k, v = (torch.cat([new[t][layer][i] for t in range(tokens)], dim=2).double() for i in range(3))
        if case.get("rope"):
            cos, sin = _rotary(x, [case["past"] + t for t in range(tokens)], case["dim"], case["dtype"])
            q, k = _rotate(q, cos, sin), _rotate(k, cos, sin)
            if store != "plain":
                k = k.to(_TORCH[case["dtype"]])   # the type that is quantised
        out = torch.empty_like(q)
        for i in range(b):
            ki, vi = (_stored(new_rows[i], store) if rows is None else torch.cat([_stored(rows[i], store), _stored(new_rows[i], store)], dim=1)
                      for rows, new_rows in zip(past[layer], (k, v)))
            out[i] = _attend(q[i], ki, vi, True)
        for t in range(tokens):
            outs[t][layer] = out[:, :, t : t + 1] if single else out
        kept += [k, v]
    return [o for per in outs for o in per] + (kept if store == "plain" else [])


def _exact_ragged(case, x):
    lens = _lengths(case, np.random.default_rng(7))
    past = list(_ragged_rows(case, x, lens))
    new = [_new_rows(case, x, case["seqs"], 1) for _ in range(case["tokens"])]
    q, k, v = (torch.cat([t[i] for t in new], dim=2) for i in range(3))
    out = torch.empty(q.shape, device="cuda", dtype=torch.float64)
    for i in range(case["seqs"]):
        ki, vi = (torch.cat([_stored(past[2 * i + j][0], case["store"]), _stored(r[i], case["store"])], dim=1) for j, r in enumerate((k, v)))
        out[i] = _attend(q[i].double(), ki, vi, True)
    return [out[:, :, t : t + 1] for t in range(case["tokens"])]


def _exact_project(case, x):
    outs = []
    for weights, act in _project_inputs(case, x):
        scale, codes = _q4_0_codes(weights)
        w = ((codes.double() - 8.0) * scale.to(torch.float16).double()).reshape(weights.shape)
        outs.append(torch.matmul(act.double(), w.t().contiguous()))
    return outs


def _exact_kivi(case, x):
    """Keys: 8-bit codes of a channel, written with the smallest value and the widest range up to their token and read with
    the newest ones; values: 8-bit codes per token.  Every token of a call sees all of the cache."""
    new = _kivi_inputs(case, x)
    k, v = (torch.cat([t[i] for t in new], dim=2).float() for i in (1, 2))
    lo = torch.cummin(k, dim=2).values
    scale = torch.cummax((k - lo) / 255.0, dim=2).values.clamp(min=1.0)
    codes = _round_half_away((k - lo) / scale).clamp(0, 255)
    vlo, vhi = v.amin(dim=3, keepdim=True), v.amax(dim=3, keepdim=True)
    vscale = torch.where(vhi > vlo, (vhi - vlo) / 255.0, torch.ones_like(vlo))
    values = vlo.double() + _round_half_away((v - vlo) / vscale).clamp(0, 255) * vscale.double()
    outs, t = [], 0
    for q, _, _ in new:
        t += q.shape[2]
        keys = lo[:, :, t - 1 : t].double() + codes[:, :, :t] * scale[:, :, t - 1 : t].double()
        outs.append(torch.stack([_attend(q[i].double(), keys[i], values[i, :, :t].contiguous(), False) for i in range(case["batch"])]))
    return outs


_EXACT = {"step": _exact_cached, "ragged": _exact_ragged, "chunk": _exact_cached, "project": _exact_project, "kivi": _exact_kivi}


def exact(case, seed):
    return _EXACT[case["kind"]](case, _Inputs(seed))


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
