"""Single tokens over numbers of sequence-heads that do not divide the compute units: one range, a few, more than the narrow
and the wide merge take."""
import ctypes as C

import numpy as np
import pytest

import tract_amd as ta
from oracle import oracle as orc
from tests.cases import textbook_sdpa
from tests.gpu_util import rt  # noqa: F401
from tract_amd._lib import call

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("store", ["plain", "Q8_0", "Q4_0"])
@pytest.mark.parametrize("B,Hq,Hkv,D,T", [(1, 8, 1, 128, 5000), (3, 32, 8, 128, 1100), (12, 8, 8, 128, 390), (28, 32, 8, 128, 129), (1, 16, 2, 128, 127),
                                           (13, 14, 2, 128, 260), (13, 8, 2, 64, 515)])
def test_steps_of_any_number_of_sequence_heads(rt, store, B, Hq, Hkv, D, T):
    if store != "plain" and D != 128:
        pytest.skip("block-quantised steps are of 128 features")
    rng = np.random.default_rng(B * 100 + T)
    k, v = (rng.standard_normal((B, Hkv, T, D), dtype=np.float32).astype(np.float16) for _ in range(2))
    q = (rng.standard_normal((B, Hq, 1, D), dtype=np.float32) / np.float32(np.sqrt(D))).astype(np.float16)
    fmt = None if store == "plain" else getattr(ta, store)
    st = ta.InPlaceKvSdpa(axis=2, causal=True, storage_format=fmt).state()
    st.k.push(k[:, :, :-1]), st.v.push(v[:, :, :-1])
    got = st.eval([q, np.ascontiguousarray(k[:, :, -1:]), np.ascontiguousarray(v[:, :, -1:])]).to_numpy().astype(np.float64)
    if fmt is not None:
        code = {"Q8_0": orc.FMT_Q8_0, "Q4_0": orc.FMT_Q4_0}[store]
        k, v = (orc.dequant(code, orc.quant(code, x), np.float32).reshape(x.shape) for x in (k, v))
    want = orc.flash_sdpa(q.astype(np.float32), k.astype(np.float32), v.astype(np.float32), causal=True, threads=8)
    # probabilities and results are rounded to f16 (2^-11 each): twice 2^-11 of the largest |v|
    assert np.abs(got - want).max() <= 2 * 2.0 ** -11 * np.abs(v.astype(np.float64)).max()


# 2 to 8 ranges, up to 32 in the kernel and more by a launch, one to sixteen heads per kv head
@pytest.mark.parametrize("B,Hq,Hkv,D,T", [(1, 32, 32, 64, 700), (6, 32, 32, 128, 700), (3, 32, 8, 128, 300), (12, 32, 8, 128, 1000), (4, 24, 8, 128, 2000), (1, 14, 2, 128, 3000),
                                           (2, 16, 1, 128, 900), (1, 8, 1, 128, 5000), (1, 32, 8, 64, 2500), (1, 64, 8, 128, 3500), (5, 14, 2, 64, 1700)])
@pytest.mark.parametrize("dtype", [np.float16, np.float32])
@pytest.mark.parametrize("where", ["first", "last", "anywhere"])
def test_an_infinite_range(rt, dtype, B, Hq, Hkv, D, T, where):
    """One token's value is infinite in a feature: so is the result there, and nowhere else, whichever range it is in."""
    rng = np.random.default_rng(T)
    q, k, v = ((0.1 if i == 0 else 1.0) * rng.standard_normal((B, h, n, D), dtype=np.float32) for i, (h, n) in enumerate([(Hq, 1), (Hkv, T), (Hkv, T)]))
    q, k, v = q.astype(dtype), k.astype(dtype), v.astype(dtype)
    for b in range(B):
        for h in range(Hkv):
            v[b, h, {"first": 0, "last": T - 2, "anywhere": rng.integers(T)}[where], 9] = np.inf
    st = ta.InPlaceKvSdpa(axis=2, causal=True).state()
    st.k.push(k[:, :, :-1]), st.v.push(v[:, :, :-1])
    got = st.eval([q, np.ascontiguousarray(k[:, :, -1:]), np.ascontiguousarray(v[:, :, -1:])]).to_numpy()
    assert np.isposinf(got[..., 9]).all() and np.isfinite(np.delete(got, 9, axis=-1)).all()


@pytest.mark.parametrize("T", [3092, 3701, 6143, 14759, 19764])
def test_more_than_eight_splits_come_in_eights(rt, T):
    """Eight sequence-heads of any length: a split's place on the XCDs is every head's.  (Seen in the records that are left in the workspace.)"""
    B, Hq, Hkv, D = 1, 32, 8, 128
    rng = np.random.default_rng(T)
    k, v = (rng.standard_normal((B, Hkv, T, D), dtype=np.float32).astype(np.float16) for _ in range(2))
    q = (rng.standard_normal((B, Hq, 1, D), dtype=np.float32) / np.float32(np.sqrt(D))).astype(np.float16)
    ws = ta.Workspace(B, Hq, 1, D)
    counters = 64 * 1024
    empty = np.concatenate([np.zeros(counters, np.uint8), np.full(ws.nbytes - counters, 0xFF, np.uint8)])
    dw = ta.DeviceTensor.from_numpy(empty)
    dq, dk, dv, out = (ta.DeviceTensor.from_numpy(x) for x in (q, k, v, np.zeros_like(q)))
    strides = (C.c_int64 * 3)(Hkv * T * D, T * D, D)
    call("trocm_sdpa", dq.ptr, dk.ptr, dv.ptr, None, out.ptr, ta.F16, B, Hq, Hkv, 1, T, D, strides, 1, 1, C.c_float(float("nan")), 1, dw.ptr, ws.nbytes, None)
    want = orc.flash_sdpa(q.astype(np.float32), k.astype(np.float32), v.astype(np.float32), causal=True, threads=8)
    assert np.abs(out.to_numpy().astype(np.float64) - want).max() <= 2 * 2.0 ** -11 * np.abs(v.astype(np.float64)).max()
    used = np.flatnonzero(dw.to_numpy()[counters:] != 0xFF).max() + 1
    record = B * Hkv * 8 * (D + 2) * 4   # of one split: rows of eight heads per kv head, their maxima and sums
    splits = -(-used // record)
    assert splits > 8 and splits % 8 == 0


# 32 heads over 8 and 64 over 8 with 64 features (f32: the matrix instruction), one head per kv head (vector units)
@pytest.mark.parametrize("dtype,B,Hq,Hkv,D,T", [(np.float32, 1, 32, 8, 128, 500), (np.float32, 2, 64, 8, 64, 900), (np.float32, 1, 32, 32, 128, 300),
                                                 (np.float32, 2, 8, 4, 64, 700), (np.float16, 1, 32, 32, 128, 300), (np.float16, 3, 16, 16, 64, 40)])
@pytest.mark.parametrize("size", [6e4, 3e10, 1e30])   # (f16: a tenth of its largest, half of it, its largest)
def test_a_key_that_is_larger_than_all_others_together(rt, dtype, B, Hq, Hkv, D, T, size):
    """A query that points along it sees that token's value alone, one that points away from it does not see the token at all."""
    if dtype is np.float16:
        size = {6e4: 6550, 3e10: 32752, 1e30: 65504}[size]
    rng = np.random.default_rng(T)
    q, k, v = (rng.standard_normal((B, h, n, D), dtype=np.float32) for h, n in [(Hq, 1), (Hkv, T), (Hkv, T)])
    first = 8 if dtype is np.float32 else D   # (f16: a score of 2^31 and more takes every feature)
    k[:, :, T // 3, :first] = size
    along = rng.integers(2, size=(B, Hq, 1, 1)) > 0
    if dtype is np.float16:
        q = np.where(along, np.float32(size), q / 4 - (q / 4).mean(axis=-1, keepdims=True) - np.float32(0.25))
    else:
        q[..., :first] = np.where(along, 1, -1) * np.abs(q[..., :first])
    q, k, v = q.astype(dtype), k.astype(dtype), v.astype(dtype)
    st = ta.InPlaceKvSdpa(axis=2, causal=True).state()
    st.k.push(k[:, :, :-1]), st.v.push(v[:, :, :-1])
    got = st.eval([q, np.ascontiguousarray(k[:, :, -1:]), np.ascontiguousarray(v[:, :, -1:])]).to_numpy().astype(np.float64)
    want = textbook_sdpa(q, k, v, causal=True)
    tol = 2 * 2.0 ** -11 if dtype is np.float16 else 2.0 ** -20   # (as above, and as the f32 steps' own tests)
    assert np.abs(got - want).max() <= tol * np.abs(v.astype(np.float64)).max()


# eight splits of which some have a group of tiles more than others
@pytest.mark.parametrize("store", ["plain", "Q8_0", "Q4_0"])
@pytest.mark.parametrize("B,Hq,Hkv,T", [(2, 32, 8, 1030), (2, 32, 8, 1500), (3, 14, 2, 2049), (2, 40, 8, 2500)])
def test_eight_unequal_splits(rt, store, B, Hq, Hkv, T):
    test_steps_of_any_number_of_sequence_heads(rt, store, B, Hq, Hkv, 128, T)
