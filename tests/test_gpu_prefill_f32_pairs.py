"""Attention of more than 32 f32 query rows, whose operands are pairs of f16 on the matrix cores: edges of its tiles, ranges of keys,
and values for which the pairs are not enough."""
import numpy as np
import pytest

import tract_amd as ta
from tests.cases import textbook_sdpa
from tests.gpu_util import rt  # noqa: F401

pytestmark = pytest.mark.gpu


def _normal(rng, *shape):
    return rng.standard_normal(shape, dtype=np.float32)


def _run(q, k, v, past, causal=True):
    st = ta.InPlaceKvSdpa(axis=2, causal=causal).state()
    if past:
        st.k.push(k[:, :, :past]), st.v.push(v[:, :, :past])
    return st.eval([q, np.ascontiguousarray(k[:, :, past:]), np.ascontiguousarray(v[:, :, past:])]).to_numpy()


# 64 rows per workgroup (q_len * group), two sets of 32-key tiles: one row more and less than a half and a whole tile of rows, keys
# around an edge of a tile and of a pair of them, ranges of keys and their merge, one tile less than the kernel takes
@pytest.mark.parametrize("B,Hq,Hkv,D,past,n", [(1, 1, 1, 128, 95, 33), (1, 2, 1, 128, 96, 16), (2, 4, 1, 64, 113, 16), (1, 5, 1, 128, 0, 129),
                                                (1, 8, 2, 128, 31, 161), (3, 3, 1, 64, 200, 43), (1, 4, 2, 128, 3001, 30), (1, 14, 2, 64, 1500, 12),
                                                (2, 32, 8, 128, 0, 300), (1, 2, 2, 128, 62, 34)])
@pytest.mark.parametrize("causal", [True, False])
def test_pairs(rt, B, Hq, Hkv, D, past, n, causal):
    rng = np.random.default_rng(B + Hq + past + n)
    q, k, v = _normal(rng, B, Hq, n, D), _normal(rng, B, Hkv, past + n, D), _normal(rng, B, Hkv, past + n, D)
    got, want = _run(q, k, v, past, causal), textbook_sdpa(q, k, v, causal=causal)
    # as the f32 kernel for fewer rows: a few 2^-24 of the norm, scores up to about 6 carry 2^-24 * 6 into the exponent
    assert np.linalg.norm(got - want) <= 2e-6 * np.linalg.norm(want)
    assert np.abs(got - want).max() <= 2e-5 * np.abs(want).max()


@pytest.mark.parametrize("what", ["tiny", "huge", "weak feature", "weak feature later", "zeros first", "larger later", "zero rows", "wide keys"])
@pytest.mark.parametrize("D", [64, 128])
def test_values_outside_the_pairs(rt, D, what):
    """Every feature of the result to f32's precision, whatever the magnitudes are."""
    rng = np.random.default_rng(D)
    past, n = 150, 70
    q, k, v = _normal(rng, 1, 4, n, D), _normal(rng, 1, 2, past + n, D), _normal(rng, 1, 2, past + n, D)
    if what == "tiny":
        q, k, v = q * np.float32(1e-20), k * np.float32(1e20), v * np.float32(1e-25)
    elif what == "huge":
        q, k, v = q * np.float32(1e10), k * np.float32(1e-10), v * np.float32(1e30)
    elif what == "weak feature":
        v[..., 7] *= np.float32(2.0 ** -22)
    elif what == "weak feature later":
        v[:, :, 100:, 7] *= np.float32(2.0 ** -10)
    elif what == "zeros first":
        k[:, :, :70], v[:, :, :70] = 0, 0
    elif what == "larger later":
        k[:, :, 180] *= 30
        v[:, :, 190:] *= 1000
    elif what == "zero rows":
        q[:, :, 3], k[:, :, 40], v[:, :, 200] = 0, 0, 0
    else:
        k[..., 3] *= 1000
        q[..., 3] /= 1000
    got, want = _run(q, k, v, past), textbook_sdpa(q, k, v, causal=True)
    for d in range(D):   # feature by feature: the bound of the whole result holds for each
        assert np.linalg.norm(got[..., d] - want[..., d]) <= 4e-6 * np.linalg.norm(want[..., d]), d


@pytest.mark.parametrize("D", [64, 128])
def test_a_later_infinity_stays_out(rt, D):
    rng = np.random.default_rng(D)
    past, n = 100, 60
    q, k, v = _normal(rng, 1, 4, n, D), _normal(rng, 1, 2, past + n, D), _normal(rng, 1, 2, past + n, D)
    v[0, 0, 140, 5], v[0, 1, past + n - 1, D - 1], v[0, 1, 133, 0] = np.inf, np.nan, -np.inf
    got = _run(q, k, v, past)
    want = textbook_sdpa(q, k, np.where(np.isfinite(v), v, 0.0), causal=True)
    for h in range(4):
        for key, d, value in ([(140, 5, np.inf)] if h < 2 else [(past + n - 1, D - 1, np.nan), (133, 0, -np.inf)]):
            want[0, h, key - past :, d] = value
    np.testing.assert_array_equal(np.isfinite(got), np.isfinite(want))
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    fine = np.isfinite(want)
    assert np.abs(got[fine] - want[fine]).max() <= 2e-5 * np.abs(want[fine]).max()
