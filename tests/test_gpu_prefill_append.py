"""Prompts and chunks of one whose new rows the attention launch reads from the call's input and stores to the cache itself: bit for
bit the attention over the same rows in one tensor, and the cache bit for bit the rows."""
import ctypes as C

import numpy as np
import pytest

import tract_amd as ta
from tests.cases import textbook_sdpa
from tests.gpu_util import rt  # noqa: F401
from tract_amd._lib import call

pytestmark = pytest.mark.gpu


def _inputs(dtype, B, Hq, Hkv, D, past, n):
    rng = np.random.default_rng(past + n)
    return tuple(rng.standard_normal((B, h, t, D), dtype=np.float32).astype(dtype) for h, t in ((Hq, n), (Hkv, past + n), (Hkv, past + n)))


def _over_one_tensor(q, k, v, causal):
    B, Hq, n, D = q.shape
    Hkv, T = k.shape[1:3]
    dq, dk, dv = (ta.DeviceTensor.from_numpy(x) for x in (q, k, v))
    out = ta.DeviceTensor(q.shape, q.dtype)
    ws = ta.Workspace(B, Hq, n, D)
    call("trocm_sdpa", dq.ptr, dk.ptr, dv.ptr, None, out.ptr, ta.F16 if q.dtype == np.float16 else ta.F32, B, Hq, Hkv, n, T, D,
         (C.c_int64 * 3)(Hkv * T * D, T * D, D), 1, 1, C.c_float(float("nan")), int(causal), ws.ptr, ws.nbytes, None)
    return out.to_numpy()


def _state(k, v, past, n, causal):
    """Caches of `past` tokens, in planes longer than they need."""
    st = ta.InPlaceKvSdpa(axis=2, causal=causal).state()
    for c, x in ((st.k, k), (st.v, v)):
        c.reserve(past + n + 37, like=((x.shape[0], x.shape[1], 1, x.shape[3]), x.dtype))
        if past:
            c.push(x[:, :, :past])
    return st


# the first new row on a tile's edge, before it and behind it, all of them in one tile; pieces that do not go round; 1 to 8 query heads
# per kv head, key splits merged by the last of them and by a launch, a workgroup alone on its unit, a last round cut into 2, 3 and 4
# ranges of keys (1, 2 and 4 query heads per workgroup); f32: none, one and many ranges of keys, one workgroup, behind whole tiles of keys
# (behind others the sums are taken in another order: below)
@pytest.mark.parametrize("dtype,B,Hq,Hkv,D,past,n", [
    (np.float16, 1, 8, 2, 128, 640, 150), (np.float16, 2, 8, 2, 128, 639, 99), (np.float16, 1, 16, 4, 128, 65, 301), (np.float16, 1, 14, 2, 128, 700, 99),
    (np.float16, 2, 4, 4, 128, 0, 700), (np.float16, 1, 32, 32, 64, 30, 1001), (np.float16, 3, 16, 2, 64, 1, 333), (np.float16, 4, 64, 8, 64, 0, 300),
    (np.float16, 1, 8, 8, 64, 2000, 70), (np.float16, 1, 32, 8, 128, 3000, 41), (np.float16, 1, 2, 1, 128, 5, 65),
    (np.float16, 2, 60, 60, 128, 1300, 530), (np.float16, 1, 128, 64, 128, 1300, 613), (np.float16, 1, 168, 42, 128, 1001, 400),
    (np.float32, 1, 8, 2, 128, 0, 150), (np.float32, 2, 14, 2, 64, 0, 171), (np.float32, 1, 32, 32, 128, 0, 333), (np.float32, 1, 6, 6, 64, 0, 1100),
    (np.float32, 1, 8, 2, 128, 0, 60), (np.float32, 1, 8, 2, 128, 64, 200)])
def test_rows_from_the_call(rt, dtype, B, Hq, Hkv, D, past, n):
    q, k, v = _inputs(dtype, B, Hq, Hkv, D, past, n)
    for causal in (True, False):
        st = _state(k, v, past, n, causal)
        for _ in range(2):   # again over what the first call left behind
            if past or _:
                st.k.truncate(past), st.v.truncate(past)
            got = st.eval([q, np.ascontiguousarray(k[:, :, past:]), np.ascontiguousarray(v[:, :, past:])]).to_numpy()
            assert st.k.valid_contiguous().tobytes() == k.tobytes() and st.v.valid_contiguous().tobytes() == v.tobytes()
            assert got.tobytes() == _over_one_tensor(q, k, v, causal).tobytes(), causal


# an output over the new keys or values (as many kv heads as query heads): appended first
@pytest.mark.parametrize("dtype,past,n", [(np.float16, 100, 200), (np.float32, 0, 200)])
@pytest.mark.parametrize("over", ["k", "v"])
def test_results_over_the_new_rows(rt, dtype, past, n, over):
    q, k, v = _inputs(dtype, 2, 4, 4, 128, past, n)
    st = _state(k, v, past, n, True)
    args = {"k": ta.DeviceTensor.from_numpy(np.ascontiguousarray(k[:, :, past:])), "v": ta.DeviceTensor.from_numpy(np.ascontiguousarray(v[:, :, past:]))}
    got = st.eval_into(ta.DeviceTensor.from_numpy(q), args["k"], args["v"], args[over]).to_numpy()
    assert st.k.valid_contiguous().tobytes() == k.tobytes() and st.v.valid_contiguous().tobytes() == v.tobytes()
    assert got.tobytes() == _over_one_tensor(q, k, v, True).tobytes()


# new rows that do not begin on a 16-byte boundary: an append launch, then the attention (a few queries on the decode tiles, a prompt, f32)
@pytest.mark.parametrize("dtype,Hq,past,n", [(np.float16, 8, 300, 3), (np.float16, 8, 300, 150), (np.float16, 8, 0, 70), (np.float32, 8, 300, 3), (np.float32, 8, 65, 150), (np.float32, 8, 0, 70)])
def test_rows_that_the_launch_does_not_take(rt, dtype, Hq, past, n):
    q, k, v = _inputs(dtype, 2, Hq, 2, 128, past, n)
    st = _state(k, v, past, n, True)

    def shifted(x):
        x = np.ascontiguousarray(x)
        whole = ta.DeviceTensor.from_numpy(np.concatenate([np.zeros(1, dtype), x.ravel()]))
        return ta.DeviceTensor(x.shape, dtype, ptr=whole.ptr.value + whole.dtype.itemsize, owner=whole)

    for _ in range(2):
        if past or _:
            st.k.truncate(past), st.v.truncate(past)
        got = st.eval_into(ta.DeviceTensor.from_numpy(q), shifted(k[:, :, past:]), shifted(v[:, :, past:])).to_numpy()
        assert st.k.len() == st.v.len() == past + n
        assert st.k.valid_contiguous().tobytes() == k.tobytes() and st.v.valid_contiguous().tobytes() == v.tobytes()
        assert got.tobytes() == _over_one_tensor(q, k, v, True).tobytes()


# f32 rows that would begin a fifth tile of keys in a range, or a range more than the units take at once, where a workgroup's four waves take four
# tiles at once: an append launch, then whole tiles
@pytest.mark.parametrize("B,Hq,Hkv,D,past,n", [(1, 40, 8, 64, 56, 71), (1, 32, 32, 128, 100, 10), (2, 32, 8, 128, 97, 3), (1, 14, 2, 64, 65, 63), (16, 32, 32, 64, 250, 4), (3, 32, 32, 128, 244, 5), (2, 32, 32, 128, 500, 5),
                                               (6, 32, 32, 64, 244, 5)])
def test_rounds_of_four_tiles_stay_full(rt, B, Hq, Hkv, D, past, n):
    q, k, v = _inputs(np.float32, B, Hq, Hkv, D, past, n)
    st = _state(k, v, past, n, True)
    got = st.eval([q, np.ascontiguousarray(k[:, :, past:]), np.ascontiguousarray(v[:, :, past:])]).to_numpy()
    assert st.k.valid_contiguous().tobytes() == k.tobytes() and st.v.valid_contiguous().tobytes() == v.tobytes()
    assert got.tobytes() == _over_one_tensor(q, k, v, True).tobytes()


# f32 rows behind a cache whose last tile of keys is not full (the call's rows begin a tile of their own): one row and all but one of a tile,
# up to 32 rows per kv head and more, ranges of keys, 1 to 8 query heads per kv head
@pytest.mark.parametrize("B,Hq,Hkv,D,past,n", [(1, 8, 2, 128, 1, 3), (2, 4, 4, 64, 31, 2), (1, 14, 2, 128, 348, 10), (3, 32, 8, 64, 801, 11), (6, 32, 8, 128, 910, 3), (1, 8, 2, 128, 33, 200),
                                               (1, 32, 8, 128, 225, 373), (2, 6, 2, 64, 1999, 65), (1, 16, 16, 128, 500, 97), (1, 64, 8, 64, 95, 33)])
@pytest.mark.parametrize("causal", [True, False])
def test_f32_rows_behind_a_cache(rt, B, Hq, Hkv, D, past, n, causal):
    q, k, v = _inputs(np.float32, B, Hq, Hkv, D, past, n)
    want = textbook_sdpa(q, k, v, causal=causal)
    for poisoned in (False, True):
        if poisoned:   # a value that only the last query sees (all of them without a causal mask), and one in the cache's last row
            v[0, 0, past + n - 1, 2], v[B - 1, Hkv - 1, past - 1, 1] = np.inf, -np.inf
        st = _state(k, v, past, n, causal)
        got = st.eval([q, np.ascontiguousarray(k[:, :, past:]), np.ascontiguousarray(v[:, :, past:])]).to_numpy().astype(np.float64)
        assert st.k.valid_contiguous().tobytes() == k.tobytes() and st.v.valid_contiguous().tobytes() == v.tobytes()
        if poisoned:
            G = Hq // Hkv
            seen = got[0, :G, :, 2] if not causal else got[0, :G, -1:, 2]
            assert np.all(np.isposinf(seen)) and np.all(np.isneginf(got[B - 1, Hq - G :, :, 1]))
            if causal:
                assert np.all(np.isfinite(got[0, :G, :-1, 2]))
            got = np.where(np.isfinite(got), got, want)
        # as many f32 roundings as additions stand one after the other, of a mean of values of about 1; measured 2e-7 of the norm
        assert np.linalg.norm(got - want) <= 1e-6 * np.linalg.norm(want)
        assert np.abs(got - want).max() <= 2e-5 * np.abs(want).max()


# the call's rows begin a tile of keys of their own: 21 and 61 tiles for 620 and 1915 tokens, in 6 and 16 ranges of four, one for each wave (in 5
# and 15 ranges one wave would take two); 45 tiles of 24 kv heads in 9 ranges of five (12 of four would be more workgroups than compute units)
@pytest.mark.parametrize("B,Hq,Hkv,past,n,ranges", [(2, 32, 8, 618, 2, 6), (1, 32, 8, 1910, 5, 16), (3, 64, 8, 1405, 4, 9)])
def test_f32_ranges_count_the_tile_that_is_not_full(rt, B, Hq, Hkv, past, n, ranges):
    q, k, v = _inputs(np.float32, B, Hq, Hkv, 128, past, n)
    st = _state(k, v, past, n, True)
    new = [ta.DeviceTensor.from_numpy(np.ascontiguousarray(x)) for x in (q, k[:, :, past:], v[:, :, past:])]
    st.eval_into(*new)   # (makes the state's workspace)
    st.k.truncate(past), st.v.truncate(past)
    call("trocm_memset", C.c_void_p(st._ws.ptr.value + 64 * 1024), 0xA5, st._ws.nbytes - 64 * 1024, None)
    got = st.eval_into(*new).to_numpy()
    kept = st._ws.buf.to_numpy()[64 * 1024 :]
    stored = ranges * B * Hkv * (32 * 128 + 64) * 4   # a range's results of up to 32 rows per kv head, their maxima and sums
    assert (kept[:stored].reshape(-1, 256) != 0xA5).any(axis=-1).all() and (kept[stored:] == 0xA5).all()
    want = textbook_sdpa(q, k, v, causal=True)
    assert np.linalg.norm(got - want) <= 1e-6 * np.linalg.norm(want)   # (as above)
