"""Single f32 tokens of grouped heads on the f32 matrix instruction, against a float64 restatement, the bytes that were appended
and the unfused sequence of operators."""
import numpy as np
import pytest

import tract_amd as ta
from oracle import oracle as orc
from tests.cases import textbook_sdpa
from tests.gpu_util import rt  # noqa: F401

pytestmark = pytest.mark.gpu


def _check(got, q, k, v):
    want = textbook_sdpa(q, k, v, causal=True)
    # a score is a sum of D products (error 2^-24 times its length in the worst case, a few of that in earnest), a result a mean
    # of rows of v under weights that are off by as much: 2^-20 of the largest |v| allows for 16 roundings in a row
    assert np.abs(got.astype(np.float64) - want).max() <= 2.0 ** -20 * np.abs(v).max()


# Groups of 3 to 16 heads (5 and more at 64 features), lengths around a tile of 16 tokens and a workgroup's four of them; one range, ranges merged in the kernel (up to 32),
# one sequence-head with more tokens than those take (the vector kernel); growth of the cache on the way
@pytest.mark.parametrize("B,Hq,Hkv,D,past", [(1, 3, 1, 128, 0), (2, 8, 2, 128, 14), (1, 5, 1, 64, 15), (1, 16, 2, 64, 16), (3, 14, 2, 128, 62), (2, 40, 8, 64, 63),
                                              (1, 16, 1, 128, 64), (4, 24, 8, 128, 250), (24, 64, 8, 128, 131), (1, 32, 2, 128, 1000), (3, 64, 8, 128, 2000),
                                              (1, 8, 1, 128, 9000), (13, 40, 8, 128, 300)])
def test_steps_of_grouped_f32_heads(rt, B, Hq, Hkv, D, past):
    rng = np.random.default_rng(Hq * 10 + past)
    k = rng.standard_normal((B, Hkv, past + 3, D), dtype=np.float32)
    v = rng.standard_normal((B, Hkv, past + 3, D), dtype=np.float32)
    st = ta.InPlaceKvSdpa(axis=2, causal=True).state()
    if past:
        st.k.push(k[:, :, :past]), st.v.push(v[:, :, :past])
    for t in range(past, past + 3):
        q = 3 * rng.standard_normal((B, Hq, 1, D), dtype=np.float32) / np.float32(np.sqrt(D))
        got = st.eval([q, np.ascontiguousarray(k[:, :, t : t + 1]), np.ascontiguousarray(v[:, :, t : t + 1])]).to_numpy()
        _check(got, q, k[:, :, : t + 1], v[:, :, : t + 1])
    assert st.k.valid_contiguous().tobytes() == k.tobytes() and st.v.valid_contiguous().tobytes() == v.tobytes()


@pytest.mark.parametrize("B,Hq,Hkv,D,past,per_sequence", [(2, 8, 2, 128, 40, True), (1, 64, 8, 128, 700, False), (3, 12, 2, 64, 15, True)])
def test_f32_steps_rotate_q_and_k_on_the_way_in(rt, B, Hq, Hkv, D, past, per_sequence):
    """The rotated key that is stored and the output are those of ApplyRope, ApplyRope, InPlaceKvSdpa, bit for bit."""
    rng = np.random.default_rng(past)
    op = ta.InPlaceKvSdpa(axis=2, causal=True)
    fused, plain = op.state(), op.state()
    k0, v0 = (rng.standard_normal((B, Hkv, past, D), dtype=np.float32) for _ in range(2))
    for st in (fused, plain):
        st.k.push(k0), st.v.push(v0)
    ks = k0
    for _ in range(3):
        q, k, v = (rng.standard_normal((B, h, 1, D), dtype=np.float32) for h in (Hq, Hkv, Hkv))
        angle = rng.uniform(-7, 7, (B if per_sequence else 1, 1, 1, D))
        cos, sin = np.cos(angle).astype(np.float32), np.sin(angle).astype(np.float32)
        got = fused.eval_rope_into(*(ta.DeviceTensor.from_numpy(a) for a in (q, k, v, cos, sin))).to_numpy()
        want = plain.eval([ta.ApplyRope().eval(q, cos, sin), ta.ApplyRope().eval(k, cos, sin), v]).to_numpy()
        ks = np.concatenate([ks, orc.apply_rope(k, cos, sin)], axis=2)
        assert fused.k.valid_contiguous().tobytes() == ks.tobytes()
        assert got.tobytes() == want.tobytes()


def test_f32_steps_over_a_ring_and_an_output_over_the_inputs(rt):
    rng = np.random.default_rng(3)
    B, Hq, Hkv, D, window = 2, 8, 2, 128, 37
    st = ta.WindowKvSdpa(axis=2, window=window).state()
    ks, vs = [], []
    for t in range(80):
        q, k, v = (rng.standard_normal((B, h, 1, D), dtype=np.float32) for h in (Hq, Hkv, Hkv))
        ks.append(k), vs.append(v)
        got = st.eval([q, k, v]).to_numpy()
        if t % 13 == 0 or t == 79:
            _check(got, q, np.concatenate(ks[-window:], 2), np.concatenate(vs[-window:], 2))
    # q and the output are the same memory
    st = ta.InPlaceKvSdpa(axis=2, causal=True).state()
    k, v = (rng.standard_normal((B, Hkv, 3001, D), dtype=np.float32) for _ in range(2))
    st.k.push(k[:, :, :3000]), st.v.push(v[:, :, :3000])
    q = rng.standard_normal((B, Hq, 1, D), dtype=np.float32)
    dq, dk, dv = (ta.DeviceTensor.from_numpy(np.ascontiguousarray(a)) for a in (q, k[:, :, 3000:], v[:, :, 3000:]))
    _check(st.eval_into(dq, dk, dv, dq).to_numpy(), q, k, v)


@pytest.mark.parametrize("B,Hq,Hkv,T", [(26, 64, 8, 1383), (1, 32, 32, 201), (16, 32, 8, 290)])
def test_rounding_of_f32_steps(rt, B, Hq, Hkv, T):
    """Long sums in one range, 64 features: 2.65e-7, 1.96e-7 and 2.0e-7 of the norm is what sixteen sums in several ranges leave (the vector kernel)."""
    rng = np.random.default_rng(T)
    q, k, v = (rng.standard_normal((B, h, n, 64), dtype=np.float32) for h, n in ((Hq, 1), (Hkv, T), (Hkv, T)))
    st = ta.InPlaceKvSdpa(axis=2, causal=True).state()
    st.k.push(k[:, :, :-1]), st.v.push(v[:, :, :-1])
    got = st.eval([q, np.ascontiguousarray(k[:, :, -1:]), np.ascontiguousarray(v[:, :, -1:])]).to_numpy()
    want = textbook_sdpa(q, k, v, causal=True)
    assert np.linalg.norm(got - want) <= {1383: 2.65e-7, 201: 1.96e-7, 290: 2.0e-7}[T] * np.linalg.norm(want)
