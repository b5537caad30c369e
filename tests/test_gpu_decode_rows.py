"""A few queries per sequence as columns of the decode tiles, new tokens read from the call's input and stored by the attention
launch, against a float64 restatement and the bytes that were appended."""
import ctypes as C

import numpy as np
import pytest

import tract_amd as ta
from oracle import oracle as orc
from tests.cases import textbook_sdpa
from tests.gpu_util import rt  # noqa: F401
from tract_amd._lib import call

pytestmark = pytest.mark.gpu


def _f16(rng, *shape):
    return rng.standard_normal(shape, dtype=np.float32).astype(np.float16)


# Rows of a kv head (group size * q_len) at 8, 16 and 32, one more than each, two and more groups of which the last overlaps
# its neighbour; lengths at and around a tile of 32 keys and four of them (one tile per wave), all new tokens, new tokens in
# two tiles; one split, splits merged in the kernel (8 rows) and by the second launch
@pytest.mark.parametrize("B,Hq,Hkv,D,past,n", [
    (1, 2, 1, 128, 0, 4), (1, 4, 4, 64, 27, 8), (2, 3, 1, 128, 31, 3), (1, 16, 2, 64, 29, 2), (2, 17, 1, 128, 300, 2),
    (1, 8, 2, 128, 1021, 8), (1, 11, 1, 128, 127, 3), (2, 14, 2, 64, 700, 5), (1, 7, 1, 128, 2000, 17), (1, 6, 2, 128, 255, 16),
    (3, 4, 4, 128, 64, 33), (16, 16, 8, 128, 600, 12), (12, 8, 8, 64, 1300, 10), (1, 5, 1, 64, 0, 64), (4, 32, 8, 128, 500, 8), (1, 32, 8, 128, 6000, 2)])
@pytest.mark.parametrize("causal", [True, False])
def test_rows_of_several_queries(rt, B, Hq, Hkv, D, past, n, causal):
    rng = np.random.default_rng(B + 10 * Hq + past + n)
    q = (_f16(rng, B, Hq, n, D) / np.float16(np.sqrt(D))).astype(np.float16) * np.float16(4)
    k, v = _f16(rng, B, Hkv, past + n, D), _f16(rng, B, Hkv, past + n, D)
    st = ta.InPlaceKvSdpa(axis=2, causal=causal).state()
    if past:
        st.k.push(k[:, :, :past]), st.v.push(v[:, :, :past])
    got = st.eval([q, np.ascontiguousarray(k[:, :, past:]), np.ascontiguousarray(v[:, :, past:])]).to_numpy().astype(np.float64)
    want = textbook_sdpa(q, k, v, causal=causal)
    # probabilities and results are rounded to f16 (2^-11): twice 2^-11 of a row's largest |v|, which its result cannot exceed
    assert np.abs(got - want).max() <= 2 * 2.0 ** -11 * np.abs(v.astype(np.float64)).max()
    assert np.linalg.norm(got - want) <= 2.0 ** -10 * np.linalg.norm(want)
    assert st.k.len() == st.v.len() == past + n
    assert st.k.valid_contiguous().tobytes() == k.tobytes()
    assert st.v.valid_contiguous().tobytes() == v.tobytes()
    # without the append, over the same cache
    again = ta.Sdpa(datum_type=np.float16, is_causal=causal).eval(q, k, v).to_numpy().astype(np.float64)
    assert np.abs(again - want).max() <= 2 * 2.0 ** -11 * np.abs(v.astype(np.float64)).max()


@pytest.mark.parametrize("fmt_name", ["Q8_0", "Q4_0"])
@pytest.mark.parametrize("B,Hq,Hkv,past,n", [(1, 4, 4, 30, 2), (2, 8, 2, 600, 4), (1, 8, 2, 1021, 8), (1, 14, 2, 700, 5), (2, 3, 1, 31, 5),
                                              (32, 5, 1, 290, 9), (6, 40, 8, 600, 4),   # odd groups of many heads, two row groups and one
                                              (1, 8, 2, 60, 4), (1, 8, 2, 61, 4)])   # 64 tokens and 65
def test_rows_over_a_quantised_cache(rt, fmt_name, B, Hq, Hkv, past, n):
    fmt = {"Q8_0": ta.Q8_0, "Q4_0": ta.Q4_0}[fmt_name]
    rng = np.random.default_rng(Hq + past + n)
    D = 128
    q = (_f16(rng, B, Hq, n, D) / np.float16(np.sqrt(D))).astype(np.float16)
    k, v = _f16(rng, B, Hkv, past + n, D), _f16(rng, B, Hkv, past + n, D)
    k[:, :, :, 5] *= np.float16(12)
    st = ta.InPlaceKvSdpa(axis=2, causal=True, storage_format=fmt).state()
    st.k.push(k[:, :, :past]), st.v.push(v[:, :, :past])
    got = st.eval([q, np.ascontiguousarray(k[:, :, past:]), np.ascontiguousarray(v[:, :, past:])]).to_numpy().astype(np.float64)
    kd, vd = (orc.dequant(fmt, orc.quant(fmt, t), np.float16) for t in (k, v))
    # as above, over the dequantised blocks
    assert np.abs(got - textbook_sdpa(q, kd, vd, causal=True)).max() <= 2 * 2.0 ** -11 * np.abs(vd.astype(np.float64)).max()
    assert st.k.valid_contiguous().tobytes() == orc.quant(fmt, k).tobytes()


def test_rows_growing_a_cache_in_steps(rt):
    """Chunks of changing length, some routed here and some to the prefill kernel, across capacity doublings."""
    rng = np.random.default_rng(11)
    B, Hq, Hkv, D = 2, 8, 2, 128
    st = ta.InPlaceKvSdpa(axis=2, causal=True).state()
    ks, vs = [], []
    for n in (3, 5, 1, 8, 40, 2, 70, 4, 1, 6):
        q = (_f16(rng, B, Hq, n, D) / np.float16(np.sqrt(D))).astype(np.float16)
        ks.append(_f16(rng, B, Hkv, n, D)), vs.append(_f16(rng, B, Hkv, n, D))
        got = st.eval([q, ks[-1], vs[-1]]).to_numpy().astype(np.float64)
        k, v = np.concatenate(ks, axis=2), np.concatenate(vs, axis=2)
        assert np.abs(got - textbook_sdpa(q, k, v, causal=True)).max() <= 2 * 2.0 ** -11 * np.abs(v.astype(np.float64)).max()
        assert st.k.valid_contiguous().tobytes() == k.tobytes()
        assert st.v.valid_contiguous().tobytes() == v.tobytes()


# 8, 16 and 32 rows per kv head and two groups; one tile, several per wave, splits; a token that only the last query sees, one in
# the middle of the new ones, one in a tile that all see; Q8_0: a value that is no number takes its block with it
@pytest.mark.parametrize("fmt,B,Hq,Hkv,D,past,n", [
    (None, 1, 2, 2, 128, 0, 6), (None, 2, 4, 2, 128, 37, 8), (None, 1, 8, 2, 128, 0, 8), (None, 1, 3, 1, 128, 1500, 8), (None, 1, 1, 1, 64, 30, 40),
    (None, 2, 4, 2, 64, 700, 6), (ta.Q8_0, 1, 2, 2, 128, 0, 6), (ta.Q8_0, 2, 4, 2, 128, 37, 8), (ta.Q8_0, 1, 3, 1, 128, 1500, 8)])
def test_rows_do_not_see_what_later_tokens_hold(rt, fmt, B, Hq, Hkv, D, past, n):
    rng = np.random.default_rng(past + n)
    q = (_f16(rng, B, Hq, n, D) / np.float16(np.sqrt(D))).astype(np.float16)
    k, v = _f16(rng, B, Hkv, past + n, D), _f16(rng, B, Hkv, past + n, D)
    v[0, 0, past + n - 1, 5], v[B - 1, Hkv - 1, past + n // 2, D - 1] = np.inf, -np.inf
    v[0, Hkv - 1, past + 1, 40] = np.nan
    if past:
        v[B - 1, 0, past // 2, 17] = np.inf
    st = ta.InPlaceKvSdpa(axis=2, causal=True, storage_format=fmt).state()
    if past:
        st.k.push(k[:, :, :past]), st.v.push(v[:, :, :past])
    else:   # the caches exist before the call: keys and values travel with it
        st.k.reserve(n, like=((B, Hkv, 1, D), np.float16)), st.v.reserve(n, like=((B, Hkv, 1, D), np.float16))
    got = st.eval([q, np.ascontiguousarray(k[:, :, past:]), np.ascontiguousarray(v[:, :, past:])]).to_numpy().astype(np.float64)
    if fmt is not None:
        with np.errstate(all="ignore"):
            k, v = (orc.dequant(fmt, orc.quant(fmt, t), np.float16) for t in (k, v))
    bad = np.repeat(~np.isfinite(v), Hq // Hkv, axis=1)
    reached = np.logical_or.accumulate(bad, axis=2)[:, :, past:]   # [B, Hq, n, D]: query i sees tokens up to past + i
    np.testing.assert_array_equal(~np.isfinite(got), reached)
    want = textbook_sdpa(q, k, np.where(np.isfinite(v), v, np.float16(0)), causal=True)
    assert np.abs(got - want)[~reached].max() <= 2 * 2.0 ** -11 * np.abs(v[np.isfinite(v)].astype(np.float64)).max()
    if fmt is None:
        assert got[0, 0, n - 1, 5] == np.inf   # (one infinity, no other term that is not finite)


@pytest.mark.parametrize("B,Hq,Hkv,D,past,n", [(1, 2, 2, 128, 0, 6), (1, 4, 2, 128, 900, 8), (2, 8, 2, 64, 40, 8), (1, 3, 1, 128, 33, 20)])
def test_rows_with_scores_that_are_no_numbers(rt, B, Hq, Hkv, D, past, n):
    rng = np.random.default_rng(past + n + 1)
    q = (_f16(rng, B, Hq, n, D) / np.float16(np.sqrt(D))).astype(np.float16)
    k, v = _f16(rng, B, Hkv, past + n, D), _f16(rng, B, Hkv, past + n, D)
    q[0, 1, 2, 7] = np.nan
    k[B - 1, 0, past + 4, 3] = np.nan
    st = ta.InPlaceKvSdpa(axis=2, causal=True).state()
    if past:
        st.k.push(k[:, :, :past]), st.v.push(v[:, :, :past])
    got = st.eval([q, np.ascontiguousarray(k[:, :, past:]), np.ascontiguousarray(v[:, :, past:])]).to_numpy().astype(np.float64)
    nan = np.zeros(got.shape, bool)
    nan[0, 1, 2] = True
    nan[B - 1, : Hq // Hkv, 4:] = True
    np.testing.assert_array_equal(np.isnan(got), nan)
    want = textbook_sdpa(np.nan_to_num(q), np.nan_to_num(k), v, causal=True)
    assert np.abs(got - want)[~nan].max() <= 2 * 2.0 ** -11 * np.abs(v.astype(np.float64)).max()


# the output over q, over the new keys and over the new values: 5 query heads per kv head in 6 groups of rows, more workgroups
# than run at once; as many kv heads as query heads, two groups
@pytest.mark.parametrize("B,Hq,Hkv,past,n", [(16, 40, 8, 300, 33), (4, 32, 32, 100, 33)])
@pytest.mark.parametrize("over", ["q", "k", "v"])
def test_rows_stored_over_the_calls_own_inputs(rt, over, B, Hq, Hkv, past, n):
    rng = np.random.default_rng(n + Hq)
    D = 128
    q = (_f16(rng, B, Hq, n, D) / np.float16(np.sqrt(D))).astype(np.float16)
    k, v = _f16(rng, B, Hkv, past + n, D), _f16(rng, B, Hkv, past + n, D)
    results = []
    for shared in (False, True):
        st = ta.InPlaceKvSdpa(axis=2, causal=True).state()
        st.k.push(k[:, :, :past]), st.v.push(v[:, :, :past])
        tensors = {"q": q, "k": k[:, :, past:], "v": v[:, :, past:]}
        args = {name: ta.DeviceTensor.from_numpy(t) for name, t in tensors.items()}
        out = ta.DeviceTensor(q.shape, np.float16)
        if shared:   # the input at the start of the output's memory
            whole = np.zeros(q.size, np.float16)
            whole[: tensors[over].size] = np.ascontiguousarray(tensors[over]).reshape(-1)
            out = ta.DeviceTensor.from_numpy(whole.reshape(q.shape))
            args[over] = ta.DeviceTensor(tensors[over].shape, np.float16, ptr=out.ptr, owner=out)
        results.append(st.eval_into(args["q"], args["k"], args["v"], out).to_numpy())
        assert st.k.valid_contiguous().tobytes() == k.tobytes() and st.v.valid_contiguous().tobytes() == v.tobytes()
    np.testing.assert_array_equal(results[1], results[0])


# no scratch, counters only, room for two ranges of keys, what the library asks for; K and V as [batch, token, head, feature]
# with 8 elements between rows; 8, 16 and 32 rows per kv head in f16, 20 f32 rows
@pytest.mark.parametrize("dtype,Hq,n", [(np.float16, 4, 4), (np.float16, 8, 4), (np.float16, 8, 8), (np.float16, 6, 23), (np.float32, 8, 5)])
@pytest.mark.parametrize("causal", [True, False])
def test_scratch_limits_and_strided_rows(rt, dtype, Hq, n, causal):
    rng = np.random.default_rng(n)
    B, Hkv, D, T, pad = 2, 2, 128, 2600, 8
    q = (rng.standard_normal((B, Hq, n, D)) / np.sqrt(D)).astype(dtype)
    kv = rng.standard_normal((2, B, T, Hkv * D + pad)).astype(dtype)
    k, v = (x[:, :, : Hkv * D].reshape(B, T, Hkv, D).transpose(0, 2, 1, 3) for x in kv)
    want = textbook_sdpa(q, k, v, causal=causal)
    dq, dk, dv = (ta.DeviceTensor.from_numpy(t) for t in (q, kv[0], kv[1]))
    row = Hkv * D + pad
    strides = (C.c_int64 * 3)(T * row, D, row)
    full = ta.Workspace(B, Hq, n, D)
    counters = 64 * 1024
    two = counters + 256 + 2 * B * Hkv * -(-Hq // Hkv * n // 32) * 32 * (D + 4) * 4
    for size in (0, counters, min(two, full.nbytes), full.nbytes):
        out = ta.DeviceTensor.from_numpy(np.full(q.shape, 7, dtype))
        call("trocm_sdpa", dq.ptr, dk.ptr, dv.ptr, None, out.ptr, ta.F16 if dtype == np.float16 else ta.F32, B, Hq, Hkv, n, T, D, strides, 1, 1,
             C.c_float(float("nan")), int(causal), full.ptr if size else None, size, None)
        got = out.to_numpy().astype(np.float64)
        # f16: as above; f32: sums of D products and 2600 weights, 2^-24 of the score in the exponent
        tol = 2 * 2.0 ** -11 * np.abs(v.astype(np.float64)).max() if dtype == np.float16 else 2e-5 * np.abs(want).max()
        assert np.abs(got - want).max() <= tol, size


# 9 to 32 rows per kv head in 2, 3 and 4 ranges of keys, which the last workgroup to arrive merges (and 5 and more: the launch), a last
# group of fewer rows, 64 features; an infinity of V in a range of its own stays one, calls repeated on the same counters
@pytest.mark.parametrize("B,Hq,Hkv,D,past,n,ranges", [(8, 32, 8, 128, 2200, 8, 4), (8, 24, 8, 128, 2300, 5, 4), (10, 32, 8, 128, 2600, 3, 3), (16, 32, 8, 64, 2700, 4, 2),
                                                      (4, 10, 2, 128, 2100, 9, 9), (11, 32, 8, 128, 2400, 3, 2), (5, 32, 32, 64, 1900, 11, 2)])
def test_ranges_merged_by_the_last_workgroup(rt, B, Hq, Hkv, D, past, n, ranges):
    rng = np.random.default_rng(past + n)
    k, v = (rng.standard_normal((B, Hkv, past + n, D), dtype=np.float32).astype(np.float16) for _ in range(2))
    q = rng.standard_normal((B, Hq, n, D), dtype=np.float32).astype(np.float16)
    v[0, 0, 7, 3] = np.inf
    st = ta.InPlaceKvSdpa(axis=2, causal=True).state()
    st.k.push(k[:, :, :past]), st.v.push(v[:, :, :past])
    kn, vn = np.ascontiguousarray(k[:, :, past:]), np.ascontiguousarray(v[:, :, past:])
    G = Hq // Hkv
    groups = -(-G * n // 32)
    record = 16 if -(-G * n // groups) <= 16 else 32   # rows of one
    for turn in range(3):
        st.k.truncate(past), st.v.truncate(past)
        if turn == 1:
            call("trocm_memset", C.c_void_p(st._ws.ptr.value + 64 * 1024), 0xA5, st._ws.nbytes - 64 * 1024, None)
        out = st.eval([q, kn, vn]).to_numpy().astype(np.float64)
        if turn == 1:   # a record of every range has been stored, none behind the last, and the counters are zero again
            kept, stored = st._ws.buf.to_numpy(), ranges * B * Hkv * groups * record * (D + 2) * 4
            assert not kept[: 4 * B * Hkv * groups].any()
            kept = kept[64 * 1024 :]
            assert (kept[stored - 4 * D : stored] != 0xA5).any() and (kept[stored:] == 0xA5).all()
        for b in (0, B - 1):
            for h in (0, Hq - 1):
                kh, vh = k[b, h // G].astype(np.float64), v[b, h // G].astype(np.float64)
                s = q[b, h].astype(np.float64) @ kh.T / np.sqrt(D)
                s[np.arange(past + n)[None, :] > past + np.arange(n)[:, None]] = -np.inf
                p = np.exp(s - s.max(axis=1, keepdims=True))
                p /= p.sum(axis=1, keepdims=True)
                if b == 0 and h // G == 0:
                    assert np.all(np.isposinf(out[b, h, :, 3])), turn
                    vh[7, 3], out[b, h, :, 3] = 0.0, (p @ np.where(np.isfinite(vh), vh, 0.0))[:, 3]
                # weights and results rounded to f16; f32 sums of D products in the scores (7 at most), of the tokens in the result
                assert np.all(np.abs(out[b, h] - p @ vh) <= 2.0 ** -9 * (p @ np.abs(vh)) + 2.0 ** -24), (turn, b, h)
