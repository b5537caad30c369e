"""Ragged steps: plans that travel with the launch and plans that are uploaded (more than 64 sequences), items of one to many tiles per wave,
tiles whose scores lie far apart, against attention in 64 bits."""
import numpy as np
import pytest

import tract_amd as ta
from oracle import oracle as orc
from tests.gpu_util import rt  # noqa: F401

pytestmark = pytest.mark.gpu


def run(fmt, Hq, Hkv, D, lens, poison=False):
    rng = np.random.default_rng(sum(lens) + Hq)
    dev, name = (None, None) if fmt == "f16" else (getattr(ta, fmt), getattr(orc, "FMT_" + fmt))
    kcs, vcs, ks, vs = [], [], [], []
    for n in lens:
        k, v = (rng.standard_normal((1, Hkv, n, D), dtype=np.float32) for _ in range(2))
        k[:, :, 32:64] *= 6.0   # one tile's scores reach far beyond the others': those end up with weights of almost nothing
        k, v = k.astype(np.float16), v.astype(np.float16)
        kc, vc = ta.InPlaceKvCache(2, dev), ta.InPlaceKvCache(2, dev)
        ks.append(k), vs.append(v), kcs.append(kc), vcs.append(vc)
    q = rng.standard_normal((len(lens), Hq, 1, D), dtype=np.float32).astype(np.float16)
    kn, vn = (rng.standard_normal((len(lens), Hkv, 1, D), dtype=np.float32).astype(np.float16) for _ in range(2))
    if poison:   # the token that head 0 of the first sequence sees most of
        top = int(np.argmax(ks[0][0, 0].astype(np.float64) @ q[0, 0, 0].astype(np.float64)))
        vs[0][0, 0, top, 5], vs[0][0, 0, top, 9] = np.inf, -np.inf
    for i in range(len(lens)):
        kcs[i].push(ks[i]), vcs[i].push(vs[i])
    out = ta.inplace_kv_sdpa_eval_ragged(*(ta.DeviceTensor.from_numpy(x) for x in (q, kn, vn)), kcs, vcs).to_numpy().astype(np.float64)
    for i, n in enumerate(lens):
        k, v = (np.concatenate([a[i], b[i:i + 1]], axis=2) for a, b in ((ks, kn), (vs, vn)))
        if name is not None:
            k, v = (orc.dequant(name, orc.quant(name, x), np.float32).reshape(x.shape) for x in (k, v))
        k, v = k[0].astype(np.float64), v[0].astype(np.float64)
        for h in range(Hq):
            kh, vh = k[h // (Hq // Hkv)], v[h // (Hq // Hkv)]
            qh = q[i, h, 0].astype(np.float64) / np.sqrt(D)
            s = kh @ qh
            p = np.exp(s - s.max())
            p /= p.sum()
            if poison and i == 0 and h // (Hq // Hkv) == 0:
                assert np.isposinf(out[i, h, 0, 5]) or h or np.isnan(out[i, h, 0, 5])
                if h == 0:
                    assert np.isposinf(out[i, 0, 0, 5]) and np.isneginf(out[i, 0, 0, 9])
                vh = np.where(np.isfinite(vh), vh, 0.0)
                keep = np.delete(np.arange(D), [5, 9])
            else:
                keep = np.arange(D)
            want, size = p @ vh, p @ np.abs(vh)
            # weights and results are rounded to f16, 2^-11 each; scores are f32 sums of D products; codes enter the products exactly,
            # the weights times the scales of their blocks are rounded once more, and what is added to the codes there, 1152 at most, leaves
            # again after f32 sums of 32 tokens a tile and a quarter of the tiles
            scores = 2 * D * 2.0 ** -24 * (np.abs(kh) @ np.abs(qh)).max()
            tol = 2.0 ** -10 + scores + (0 if name is None else 2.0 ** -10)
            shift = 0 if name is None else 1152 * 2.0 ** -24 * (32 + n / 128) * np.abs(vh).max() / (127 if fmt == "Q8_0" else 8)
            assert np.all(np.abs(out[i, h, 0] - want)[keep] <= (tol * size + shift + 2.0 ** -24)[keep]), (i, n, h)


SHORT = [1 + (37 * i) % 290 for i in range(65)]


@pytest.mark.parametrize("fmt", ["f16", "Q8_0", "Q4_0"])
@pytest.mark.parametrize("Hq,Hkv,lens", [(8, 2, SHORT[:64]), (8, 2, SHORT), (4, 1, [9000, 1, 33]), (16, 2, [3000, 127, 128, 129]), (10, 2, [31, 32, 1000, 5000])])
def test_plans_and_items(rt, fmt, Hq, Hkv, lens):
    run(fmt, Hq, Hkv, 128, lens)


@pytest.mark.parametrize("Hq,Hkv,lens", [(8, 2, SHORT), (14, 2, [4000, 64, 65]), (12, 1, [700, 2500]), (2, 2, [300, 40])])
def test_plans_and_items_of_64_features(rt, Hq, Hkv, lens):
    run("f16", Hq, Hkv, 64, lens)


def test_an_infinite_value_stays_one(rt):
    run("f16", 8, 2, 128, [700, 90, 2100], poison=True)
