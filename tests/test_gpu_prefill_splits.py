"""f16 prompts whose keys are split over workgroups: every way the parts are merged (by the last of up to four, by a launch for up
to eight and up to sixteen), one and two workgroups on a compute unit at head size 64, one head per workgroup with few queries, small
scratch, and what the kernel without parts takes."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

import tract_amd as ta
from tests.cases import textbook_sdpa
from tests.gpu_util import rt  # noqa: F401
from tract_amd._lib import call

pytestmark = pytest.mark.gpu

# q, K and V are exact.  A weight, a part's output and the output are rounded to f16, 2^-11 of each at most, and so is their
# root mean square over the output; the sum of three, and scores of a few units with 2^-24 each
TOL = 3 * 2.0 ** -11


def _normal(rng, *shape):
    return rng.standard_normal(shape, dtype=np.float32).astype(np.float16)


def _sdpa(q, k, v, causal, ws, size):
    B, Hq, n, D = q.shape
    Hkv, T = k.shape[1:3]
    dq, dk, dv = (ta.DeviceTensor.from_numpy(x) for x in (q, k, v))
    out = ta.DeviceTensor.from_numpy(np.full(q.shape, 7, np.float16))
    strides = (C.c_int64 * 3)(Hkv * T * D, T * D, D)
    call("trocm_sdpa", dq.ptr, dk.ptr, dv.ptr, None, out.ptr, ta.F16, B, Hq, Hkv, n, T, D, strides, 1, 1, C.c_float(float("nan")),
         int(causal), ws.ptr if size else None, size, None)
    return out.to_numpy()


@pytest.mark.parametrize("B,Hq,Hkv,D,past,n", [(1, 8, 2, 128, 3584, 65), (1, 14, 2, 128, 700, 99), (2, 5, 1, 128, 1000, 150),
                                                (1, 8, 8, 64, 2000, 120), (1, 32, 8, 64, 500, 300), (2, 14, 2, 64, 0, 700),
                                                (1, 7, 1, 64, 900, 255), (1, 32, 8, 128, 1000, 301), (3, 16, 4, 128, 0, 500),
                                                (2, 36, 12, 64, 60, 1100), (1, 32, 32, 128, 0, 70), (1, 1, 1, 64, 4000, 190)])
def test_parts(rt, B, Hq, Hkv, D, past, n):
    rng = np.random.default_rng(past + n)
    q, k, v = _normal(rng, B, Hq, n, D), _normal(rng, B, Hkv, past + n, D), _normal(rng, B, Hkv, past + n, D)
    ws = ta.Workspace(B, Hq, n, D)
    for causal in (True, False):
        want = textbook_sdpa(q, k, v, causal=causal).astype(np.float64)
        for size in ((0, 64 * 1024 + 256, ws.nbytes // 3, ws.nbytes, ws.nbytes) if causal else (ws.nbytes,)):   # (the last again: counters are left as they were)
            got = _sdpa(q, k, v, causal, ws, size).astype(np.float64)
            assert np.linalg.norm(got - want) <= TOL * np.linalg.norm(want), (causal, size)
            rows, err = np.linalg.norm(want, axis=-1), np.linalg.norm(got - want, axis=-1)
            assert (err <= 2 * TOL * rows + 2.0 ** -20).all(), (causal, size)   # row by row: none is missing or another's


# head size 64: as many workgroups of 64 queries as compute units (256), more that find place behind each other (320, one or all queries
# in the last tile), more that share a unit (behind 300 tokens, or of equal length)
@pytest.mark.parametrize("past,n,causal", [(0, 256, True), (0, 257, True), (0, 320, True), (40, 299, True), (300, 300, True), (0, 300, False)])
def test_a_compute_unit_alone_and_shared(rt, past, n, causal):
    rng = np.random.default_rng(past + n)
    q, k, v = _normal(rng, 4, 64, n, 64), _normal(rng, 4, 8, past + n, 64), _normal(rng, 4, 8, past + n, 64)
    ws = ta.Workspace(4, 64, n, 64)
    got, want = _sdpa(q, k, v, causal, ws, ws.nbytes).astype(np.float64), textbook_sdpa(q, k, v, causal=causal)
    assert np.linalg.norm(got - want) <= TOL * np.linalg.norm(want)
    assert (np.linalg.norm(got - want, axis=-1) <= 2 * TOL * np.linalg.norm(want, axis=-1) + 2.0 ** -20).all()


# 15 and 6 parts, merged by a launch; 2, 3 and 4, merged by the last of them
@pytest.mark.parametrize("heads,kv,n,past", [(8, 2, 65, 3583), (14, 2, 99, 669), (32, 8, 700, 324), (32, 8, 300, 276), (40, 8, 500, 204), (32, 8, 300, 212)])
@pytest.mark.parametrize("last", [False, True])
def test_an_infinite_part(rt, heads, kv, n, past, last):
    """One part's output is infinite in a feature: so is the result there, and nowhere else, whichever part it is.  (Whole tiles of keys.)"""
    rng = np.random.default_rng(n)
    q, k, v = _normal(rng, 1, heads, n, 128), _normal(rng, 1, kv, past + n, 128), _normal(rng, 1, kv, past + n, 128)
    q *= np.float16(0.125)   # no weight is below f16's smallest
    v[:, :, past + n - 1 if last else 0, 9] = np.inf
    ws = ta.Workspace(1, heads, n, 128)
    got = _sdpa(q, k, v, False, ws, ws.nbytes)
    assert np.isposinf(got[..., 9]).all() and np.isfinite(np.delete(got, 9, axis=-1)).all()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("T", [120, 200])
def test_short_prompts_of_odd_groups_sum_their_weights_in_f32(rt, D, T):
    """One key of weight 1 and value c, T - 1 of weight w and value 0: c / (1 + (T - 1) w), correctly rounded but for f32's own errors.
    w is half way between two f16 numbers, so that a sum of rounded weights is off by 2^-12 and more, which is another f16 number."""
    t = np.arange(2048, dtype=np.int64) / 1024 + 1.0   # f16 numbers from 1 to 3
    w = np.exp(-t)
    t, w = max(zip(t, w), key=lambda x: abs(float(np.float16(x[1])) - x[1]) / x[1])
    exact, off = 1 / (1 + (T - 1) * w), 1 / (1 + (T - 1) * float(np.float16(w)))
    # c such that c * exact lies beside a middle between two f16 numbers, on its side of it, and c * off on the other
    c = max((np.float64(x) for x in np.arange(1024, 2048) / 1024 if np.float16(x * exact) != np.float16(x * off)),
            key=lambda x: abs(np.float64(np.float16(x * exact)) - x * off) - abs(np.float64(np.float16(x * exact)) - x * exact))
    q, k, v = np.zeros((1, 14, 70, D), np.float16), np.zeros((1, 2, T, D), np.float16), np.zeros((1, 2, T, D), np.float16)
    q[..., 0], k[..., 0] = 1, -t
    k[:, :, T // 3], v[:, :, T // 3] = 0, c
    ws = ta.Workspace(1, 14, 70, D)
    B, Hq, n, _ = q.shape
    dq, dk, dv = (ta.DeviceTensor.from_numpy(x) for x in (q, k, v))
    out = ta.DeviceTensor.from_numpy(np.zeros_like(q))
    strides = (C.c_int64 * 3)(2 * T * D, T * D, D)
    call("trocm_sdpa", dq.ptr, dk.ptr, dv.ptr, None, out.ptr, ta.F16, B, Hq, 2, n, T, D, strides, 1, 1, C.c_float(1.0), 0, ws.ptr, ws.nbytes, None)
    np.testing.assert_array_equal(out.to_numpy(), np.full_like(q, np.float16(c * exact)))


@pytest.mark.parametrize("heads,kv,D,n,T", [(40, 8, 128, 70, 370), (14, 2, 64, 70, 970), (5, 5, 128, 100, 100)])
@pytest.mark.parametrize("size", [500, 20000, 60000])
def test_a_key_that_is_larger_than_all_others_together(rt, heads, kv, D, n, T, size):
    """Scores up to 2^36: queries that point along it see that token's value alone."""
    rng = np.random.default_rng(T)
    q, k, v = np.full((1, heads, n, D), size, np.float16), _normal(rng, 1, kv, T, D), _normal(rng, 1, kv, T, D)
    k[:, :, T // 3] = size
    ws = ta.Workspace(1, heads, n, D)
    got = _sdpa(q, k, v, False, ws, ws.nbytes)
    np.testing.assert_array_equal(got, np.broadcast_to(np.repeat(v[:, :, T // 3 : T // 3 + 1], heads // kv, axis=1), q.shape))


# scales that are not positive, an output that is aligned to 8 bytes only: the smaller kernel (sdpa_prefill.hip), its keys
# over two sets of waves, 64 or (from 256 workgroups on) 128 queries per workgroup
@pytest.mark.parametrize("what", ["negative scale", "zero scale", "output"])
@pytest.mark.parametrize("B,Hq,Hkv,D,past,n", [(1, 6, 2, 128, 31, 65), (1, 5, 5, 64, 0, 130), (2, 64, 8, 64, 70, 129), (1, 3, 1, 128, 300, 64)])
def test_what_only_the_smaller_kernel_takes(rt, what, B, Hq, Hkv, D, past, n):
    rng = np.random.default_rng(past + n)
    T = past + n
    q, k, v = _normal(rng, B, Hq, n, D), _normal(rng, B, Hkv, T, D), _normal(rng, B, Hkv, T, D)
    scale = {"negative scale": -0.11, "zero scale": 0.0, "output": 0.11}[what]
    at = 4 if what == "output" else 0
    ws = ta.Workspace(B, Hq, n, D)
    dq, dk, dv = (ta.DeviceTensor.from_numpy(x) for x in (q, k, v))
    strides = (C.c_int64 * 3)(Hkv * T * D, T * D, D)
    for causal in (True, False):
        out = ta.DeviceTensor.from_numpy(np.full(q.size + 8, 7, np.float16))
        call("trocm_sdpa", dq.ptr, dk.ptr, dv.ptr, None, C.c_void_p(out.ptr.value + 2 * at), ta.F16, B, Hq, Hkv, n, T, D, strides, 1, 1, C.c_float(scale), int(causal),
             ws.ptr, ws.nbytes, None)
        flat = out.to_numpy()
        assert (flat[:at] == 7).all() and (flat[at + q.size :] == 7).all()
        got, want = flat[at : at + q.size].reshape(q.shape).astype(np.float64), textbook_sdpa(q, k, v, scale=scale, causal=causal)
        assert np.linalg.norm(got - want) <= TOL * np.linalg.norm(want), causal
        assert (np.linalg.norm(got - want, axis=-1) <= 2 * TOL * np.linalg.norm(want, axis=-1) + 2.0 ** -20).all(), causal


# more query tiles than whole rounds of compute units take: those left over are cut into 2, 3 and 4 ranges of keys (one head of a
# group of one, a group of two and of four per workgroup; causal behind past tokens or unmasked; the last tile with few queries)
CUT = [(1, 384, 96, 1100, 130, True, 96, 2), (2, 160, 40, 900, 220, False, 80, 2), (1, 128, 64, 1300, 613, True, 64, 3), (2, 60, 60, 1300, 530, False, 120, 2),
       (1, 168, 42, 1000, 400, True, 42, 4)]


@pytest.mark.parametrize("store", [None, ta.Q8_0, ta.Q4_0])
@pytest.mark.parametrize("B,Hq,Hkv,past,n,causal,left,parts", CUT)
def test_tiles_left_for_the_last_round(rt, store, B, Hq, Hkv, past, n, causal, left, parts):
    rng = np.random.default_rng(n)
    T, G = past + n, Hq // Hkv
    q, k, v = _normal(rng, B, Hq, n, 128), _normal(rng, B, Hkv, T, 128), _normal(rng, B, Hkv, T, 128)
    if store is None:
        v[0, 1, 40, 9] = np.inf   # one range's output, in one feature of one kv head
    kc, vc = ta.InPlaceKvCache(2, store), ta.InPlaceKvCache(2, store)
    kc.push(k), vc.push(v)
    dq, out = ta.DeviceTensor.from_numpy(q), ta.DeviceTensor(q.shape, np.float16)
    ws = ta.Workspace(B, Hq, n, 128)
    results = []
    call("trocm_memset", C.c_void_p(ws.ptr.value + 64 * 1024), 0xA5, ws.nbytes - 64 * 1024, None)
    for size in (64 * 1024, ws.nbytes, ws.nbytes):   # whole; cut; the same bits again
        call("trocm_sdpa_cached", dq.ptr, ta.F16, Hq, n, kc._h, vc._h, out.ptr, C.c_float(float("nan")), int(causal), ws.ptr, size, None)
        results.append(out.to_numpy())
    assert results[1].tobytes() == results[2].tobytes()
    # all but one part of a tile have been stored, 8 waves' 32 x 128 sums each: the first of every tile's places, and none behind the last
    kept = ws.buf.to_numpy()[64 * 1024 :][: 16 * 1024 * 8 * left * (parts - 1)].reshape(parts - 1, left, 8, 16 * 1024)
    assert (kept[:, :, 0] != 0xA5).any(axis=-1).all()
    behind = ws.buf.to_numpy()[64 * 1024 + (parts - 1) * left * 8 * (16 * 1024 + 256) :]
    assert behind.size and (behind == 0xA5).all()
    infinite = np.zeros(q.shape, bool)
    if store is None:
        infinite[0, G : 2 * G, :, 9] = True
    for r in results[:2]:
        np.testing.assert_array_equal(np.isposinf(r), infinite)
    whole, cut = (np.where(infinite, 0, r).astype(np.float64) for r in results[:2])
    err, rows = np.linalg.norm(cut - whole, axis=-1), np.linalg.norm(whole, axis=-1)
    assert (err <= 3 * TOL * rows + 2.0 ** -20).all()   # both round as above
    if store is None:   # the first and the last heads against f64
        for b, h in ((0, 0), (B - 1, Hkv - 1)):
            want = textbook_sdpa(q[b : b + 1, h * G : (h + 1) * G], k[b : b + 1, h : h + 1], v[b : b + 1, h : h + 1], causal=causal)
            assert np.linalg.norm(cut[b, h * G : (h + 1) * G] - want[0]) <= TOL * np.linalg.norm(want)


def test_a_cut_over_counters_that_are_not_zero_ends(rt):
    """A workspace whose header is not what trocm_sdpa_workspace_init left: no part of a tile is the first to arrive, nothing is stored, and all
    of them stop waiting for it.  After another init the workspace serves again."""
    B, Hq, Hkv, past, n, causal, _, _ = CUT[0]
    rng = np.random.default_rng(1)
    q, k, v = _normal(rng, B, Hq, n, 128), _normal(rng, B, Hkv, past + n, 128), _normal(rng, B, Hkv, past + n, 128)
    kc, vc = ta.InPlaceKvCache(2), ta.InPlaceKvCache(2)
    kc.push(k), vc.push(v)
    dq, out, ws = ta.DeviceTensor.from_numpy(q), ta.DeviceTensor(q.shape, np.float16), ta.Workspace(B, Hq, n, 128)

    def run():
        call("trocm_sdpa_cached", dq.ptr, ta.F16, Hq, n, kc._h, vc._h, out.ptr, C.c_float(float("nan")), int(causal), ws.ptr, ws.nbytes, None)
        return out.to_numpy().tobytes()

    want = run()
    call("trocm_memset", ws.ptr, 0x40, 64 * 1024, None)
    run()
    call("trocm_sdpa_workspace_init", ws.ptr, ws.nbytes, None)
    assert run() == want


def test_no_merge_by_the_last_to_arrive_means_no_cut():
    """TROCM_PREFILL_TAIL_MERGE=0 (no workgroup waits for or merges another's results) leaves a last round as whole as
    TROCM_PREFILL_PARTS=0 does: the same bits, others than those of the cut."""
    code = """
import sys; sys.path.insert(0, %r)
import numpy as np, tract_amd as ta
ta.runtime_for_name("rocm")
rng = np.random.default_rng(5)
q, k, v = (rng.standard_normal((1, h, n, 128), dtype=np.float32).astype(np.float16) for h, n in ((168, 400), (42, 1400), (42, 1400)))
sys.stdout.buffer.write(ta.Sdpa(datum_type=np.float16, is_causal=True).eval(q, k, v).to_numpy().tobytes())
""" % os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

    def run(**env):
        p = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, **env), capture_output=True, timeout=100)
        assert p.returncode == 0, p.stderr[-2000:]
        return p.stdout[-168 * 400 * 128 * 2 :]

    cut, whole = run(), run(TROCM_PREFILL_PARTS="0")
    assert run(TROCM_PREFILL_TAIL_MERGE="0") == whole != cut
