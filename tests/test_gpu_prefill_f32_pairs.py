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


def _late(rng, heads, kv, past, n, D):
    """Queries that weigh the keys from 64 on only (scores 24 against -24)."""
    q, k, v = _normal(rng, 1, heads, n, D), _normal(rng, 1, kv, past + n, D), _normal(rng, 1, kv, past + n, D)
    q[..., 0], k[..., 0] = 4 * np.sqrt(D), 6
    k[:, :, :64, 0] = -6
    return q, k, v


# what starts beyond the first tiles of a range, where V's scale was taken; 30 queries behind 3000 tokens: many ranges of keys
@pytest.mark.parametrize("what", ["weak later", "weaker later", "gone later", "feature later", "weaker feature later", "feature of few keys",
                                  "first row weak", "wide channels", "wide channels later", "zero values", "values later"])
@pytest.mark.parametrize("D,past,n", [(64, 150, 70), (128, 150, 70), (128, 0, 220), (128, 3000, 30)])
def test_values_that_change_along_the_keys(rt, D, past, n, what):
    """Every feature and every row of the result to f32's precision, wherever the magnitudes change."""
    rng = np.random.default_rng(D + past)
    heads, kv, T = 4, 2, past + n
    if what in ("weak later", "weaker later", "gone later"):
        q, k, v = _late(rng, heads, kv, past, n, D)
        v[:, :, 64:] *= np.float32({"weak later": 1e-8, "weaker later": 1e-10, "gone later": 1e-16}[what])
    else:
        q, k, v = _normal(rng, 1, heads, n, D), _normal(rng, 1, kv, T, D), _normal(rng, 1, kv, T, D)
    if what in ("feature later", "weaker feature later"):
        v[:, :, :70, 7] = 0
        v[:, :, 70:, 7] *= np.float32(2.0 ** (-20 if what == "feature later" else -26))
    elif what == "feature of few keys":   # strong in the first 64, which these queries hardly weigh
        q, k, v = _late(rng, heads, kv, past, n, D)
        v[:, :, 64:, 9] *= np.float32(2.0 ** -24)
    elif what == "first row weak":
        v[:, :, 0] *= np.float32(1e-9)
    elif what == "wide channels":
        q[..., [3, 11, 40, 41]] *= 20
        k[..., [3, 11, 40, 41]] *= 20
    elif what == "wide channels later":
        k[:, :, 130:, 5] *= 200
    elif what == "zero values":
        v[:] = 0
    elif what == "values later":
        v[:, :, :130] = 0
    got, want = _run(q, k, v, past).astype(np.float64), textbook_sdpa(q.astype(np.float64), k.astype(np.float64), v.astype(np.float64), causal=True)
    # A score is a sum of D products of the size |q| |k| scale at most, rounded D times by 2^-25 of that: sqrt(D) of them in each weight
    # and again in their sum.  Over many rows and keys of scores that are alike this averages out, and a few 2^-24 remain; not in a
    # single row, nor where one product makes up every score.
    row = max(4e-6, 2 * np.sqrt(D) * 2.0 ** -25 * np.linalg.norm(q, axis=-1).max() * np.linalg.norm(k, axis=-1).max() / np.sqrt(D))
    feature = 4e-6 if np.abs(q).max() < 6 and np.abs(k).max() < 6 else row
    err = got - want
    for d in range(D):
        assert np.linalg.norm(err[..., d]) <= feature * np.linalg.norm(want[..., d]), d
    assert (np.linalg.norm(err, axis=-1) <= row * np.linalg.norm(want, axis=-1)).all()


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


# ranges of keys for up to 32 rows and for more of them
@pytest.mark.parametrize("heads,kv,D,past,n", [(8, 2, 128, 1500, 4), (4, 4, 64, 700, 20), (8, 2, 128, 1500, 20), (14, 2, 64, 1500, 12), (4, 2, 128, 3001, 60)])
@pytest.mark.parametrize("last", [False, True])
def test_an_infinite_range(rt, heads, kv, D, past, n, last):
    """One token's value is infinite in a feature: so is the result there, and nowhere else, whichever range it is in."""
    rng = np.random.default_rng(past)
    q, k, v = _normal(rng, 1, heads, n, D) / 10, _normal(rng, 1, kv, past + n, D), _normal(rng, 1, kv, past + n, D)
    v[:, :, past + n - 1 if last else 0, 9] = np.inf
    got = _run(q, k, v, past, causal=False)
    assert np.isposinf(got[..., 9]).all() and np.isfinite(np.delete(got, 9, axis=-1)).all()
