"""Attention of many f32 query rows (the f32 matrix-instruction kernel) against a float64 restatement."""
import numpy as np
import pytest

import tract_amd as ta
from tests.cases import textbook_sdpa
from tests.gpu_util import rt  # noqa: F401

pytestmark = pytest.mark.gpu


def _normal(rng, *shape):
    return rng.standard_normal(shape, dtype=np.float32)


# rows per tile 32 (q_len * group), tiles of 32 keys, 4 waves per tile: one row to several tiles, keys one before and after
# an edge, groups that do not divide 32, few rows over many keys (ranges of keys and their merge)
@pytest.mark.parametrize("B,Hq,Hkv,D,past,n", [
    (1, 1, 1, 128, 0, 2), (1, 1, 1, 64, 0, 31), (2, 4, 4, 64, 0, 33), (1, 8, 2, 128, 0, 129), (1, 5, 1, 128, 7, 13), (2, 14, 2, 64, 30, 67),
    (1, 32, 8, 128, 127, 6), (3, 8, 1, 64, 129, 5), (2, 4, 2, 128, 2047, 3), (1, 2, 1, 64, 5000, 2), (1, 40, 8, 128, 1, 96)])
@pytest.mark.parametrize("causal", [True, False])
def test_prefill_f32(rt, B, Hq, Hkv, D, past, n, causal):
    rng = np.random.default_rng(B * 1000 + Hq * 100 + past + n)
    q, k, v = _normal(rng, B, Hq, n, D), _normal(rng, B, Hkv, past + n, D), _normal(rng, B, Hkv, past + n, D)
    st = ta.InPlaceKvSdpa(axis=2, causal=causal).state()
    if past:
        st.k.push(k[:, :, :past]), st.v.push(v[:, :, :past])
    got = st.eval([q, np.ascontiguousarray(k[:, :, past:]), np.ascontiguousarray(v[:, :, past:])]).to_numpy()
    want = textbook_sdpa(q, k, v, causal=causal)
    # f32 sums of at most D products and len probabilities: a few 2^-24 of the result's norm; scores up to about 6 in
    # magnitude carry 2^-24 * 6 into the exponent
    assert np.linalg.norm(got - want) <= 2e-6 * np.linalg.norm(want)
    assert np.abs(got - want).max() <= 2e-5 * np.abs(want).max()


@pytest.mark.parametrize("D", [64, 128])
def test_prefill_f32_a_later_infinity_stays_out(rt, D):
    """A query does not see what a later key holds: V rows with infinities and NaN reach exactly the rows that see them."""
    rng = np.random.default_rng(D)
    n = 70
    q, k, v = _normal(rng, 1, 4, n, D), _normal(rng, 1, 2, n, D), _normal(rng, 1, 2, n, D)
    v[0, 0, 40, 5], v[0, 1, n - 1, D - 1], v[0, 1, 33, 0] = np.inf, np.nan, -np.inf
    got = ta.InPlaceKvSdpa(axis=2, causal=True).state().eval([q, k, v]).to_numpy()
    want = textbook_sdpa(q, k, np.where(np.isfinite(v), v, 0.0), causal=True)
    for h in range(4):
        for key, d, value in ([(40, 5, np.inf)] if h < 2 else [(n - 1, D - 1, np.nan), (33, 0, -np.inf)]):
            want[0, h, key:, d] = value
    np.testing.assert_array_equal(np.isfinite(got), np.isfinite(want))
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    fine = np.isfinite(want)
    assert np.abs(got[fine] - want[fine]).max() <= 2e-5 * np.abs(want[fine]).max()
