"""Q4_0 weights x f16 rows on the tiled matrix-matrix kernel: each of the shapes that its rule chooses, with remainders of rows and of
weight rows, against the product in 64 bits with the dequantised weights."""
import os
import subprocess
import sys

import numpy as np
import pytest

import tract_amd as ta
from oracle import oracle as orc
from tests.gpu_util import rt  # noqa: F401

pytestmark = pytest.mark.gpu


# (n, k, m): 32 rows x 128 of a tall matrix, 32 rows x 32 with k shared by 8 waves, 32 x 64 by 4 sets, 64 x 64 by 4, 64 x 128 by 4 and 2, 64 x 256 by 2, 128 x 256; odd tile
# counts (k / 128 = 3, 9, 6, 12) that only some of them or none take
@pytest.mark.parametrize("n,k,m", [(65552, 512, 31), (4096, 1024, 49), (2816, 1024, 131), (2832, 1024, 299), (4112, 1024, 321), (5120, 512, 388), (4096, 1024, 1000),
                                   (14336, 512, 390), (1040, 384, 200), (2064, 1152, 77), (3072, 768, 150), (4096, 1536, 65)])
def test_shapes_of_the_tiled_product(rt, n, k, m):
    rng = np.random.default_rng(n + k + m)
    w = (0.03 * rng.standard_normal((n, k), dtype=np.float32)).astype(np.float32)
    act = rng.standard_normal((1, m, k), dtype=np.float32).astype(np.float16)
    blocks = orc.quant(orc.FMT_Q4_0, w)
    got = ta.GgmlGemm().eval(ta.DeviceTensor.from_numpy(act), ta.Q40Weights(blocks, 1, n, k)).to_numpy().astype(np.float64)[0]
    want = act[0].astype(np.float64) @ orc.dequant(orc.FMT_Q4_0, blocks, np.float32).reshape(n, k).astype(np.float64).T
    # every weight and the result are rounded to f16 once: 2^-11 of each at most, about 0.3 of that in the norm
    assert np.linalg.norm(got - want) <= 2.0 ** -11 * np.linalg.norm(want)
    # a result is a sum of k products whose weights are off by 2^-11 at most: 6 standard deviations of that, and its own rounding
    assert np.abs(got - want).max() <= 2.0 ** -11 * (6 * np.sqrt(k) * 0.03 + np.abs(want).max())


# a tile that is given from outside in one direction only: the rest follows from it, not from the shape that would have been chosen
@pytest.mark.parametrize("given", ["BM=128", "NI=2", "NW=4", "KS=4"])
def test_a_tile_given_in_part(rt, given):
    code = """
import sys; sys.path.insert(0, %r)
import numpy as np, tract_amd as ta
from oracle import oracle as orc
ta.runtime_for_name("rocm")
rng = np.random.default_rng(0)
for n, k, m in [(4096, 1024, 49), (2816, 1024, 131), (4096, 4096, 260)]:   # chosen: 8, 4 and 4 sets of waves
    blocks = orc.quant(orc.FMT_Q4_0, (0.03 * rng.standard_normal((n, k), dtype=np.float32)).astype(np.float32))
    act = rng.standard_normal((1, m, k), dtype=np.float32).astype(np.float16)
    got = ta.GgmlGemm().eval(ta.DeviceTensor.from_numpy(act), ta.Q40Weights(blocks, 1, n, k)).to_numpy().astype(np.float64)[0]
    want = act[0].astype(np.float64) @ orc.dequant(orc.FMT_Q4_0, blocks, np.float32).reshape(n, k).astype(np.float64).T
    assert np.linalg.norm(got - want) <= 2.0 ** -11 * np.linalg.norm(want), (n, k, m)
""" % os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    name, value = given.split("=")
    p = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, **{"TROCM_Q4_MATMUL_" + name: value}), capture_output=True, text=True, timeout=100)
    assert p.returncode == 0, p.stderr[-2000:]


# the sets of waves walk 1 to 7 tiles of k each (fewer than, as many as and more than are on their way at a time, and none behind the
# last): the shapes of 32, 64 and 64 rows in 8 or 4, 4 and 2 sets
@pytest.mark.parametrize("n,m,tiles", [(n, m, t) for n, m in [(2816, 49), (2816, 131), (2832, 299), (5136, 388)] for t in (4, 8, 12, 16, 20, 24, 28)] +
                         # ... and one or two sets of one or two waves, of 32 and 64 rows, with one to three tiles, and with more
                         [(n, m, t) for n, m in [(2416, 616), (3072, 150), (12016, 32), (5008, 40)] for t in (1, 2, 3, 6, 7, 10)])
def test_short_walks_of_k(rt, n, m, tiles):
    rng = np.random.default_rng(n + tiles)
    k = 128 * tiles
    blocks = orc.quant(orc.FMT_Q4_0, (0.03 * rng.standard_normal((n, k), dtype=np.float32)).astype(np.float32))
    act = rng.standard_normal((1, m, k), dtype=np.float32).astype(np.float16)
    got = ta.GgmlGemm().eval(ta.DeviceTensor.from_numpy(act), ta.Q40Weights(blocks, 1, n, k)).to_numpy().astype(np.float64)[0]
    want = act[0].astype(np.float64) @ orc.dequant(orc.FMT_Q4_0, blocks, np.float32).reshape(n, k).astype(np.float64).T
    assert np.linalg.norm(got - want) <= 2.0 ** -11 * np.linalg.norm(want)   # (as above)
    assert np.abs(got - want).max() <= 2.0 ** -11 * (6 * np.sqrt(k) * 0.03 + np.abs(want).max())


# f32 rows: 16 x 32, 16 x 48, 16 x 64, 32 x 64, 32 x 96 and 32 x 128 (activation rows x weight rows) of tiles, 16 x 16, 16 x 32, 32 x 32, 32 x
# 64, 32 x 96 and 64 x 64 of planes, with remainders of both; one row's values are so large that its blocks are done in f32, for every part
# of the workgroup's weight rows
@pytest.mark.parametrize("m,n,k", [(16, 4130, 160), (16, 4112, 256), (64, 2817, 1056), (64, 2064, 1152), (33, 4130, 160), (33, 4112, 384), (150, 2063, 1024),
                                   (150, 2064, 1152), (150, 4100, 1056), (150, 4112, 1152), (200, 4130, 160), (200, 4112, 256),
                                   (40, 1001, 96), (130, 1001, 1056), (250, 1001, 160), (210, 4090, 544), (97, 8210, 1120),
                                   # ... and the fewest rows it takes, of small and tall matrices
                                   (5, 4112, 384), (5, 2065, 160), (6, 1040, 2176), (6, 30000, 128), (7, 57360, 128), (8, 32784, 512), (12, 65552, 256)])
def test_shapes_of_the_f32_product(rt, m, n, k):
    rng = np.random.default_rng(n + k + m)
    blocks = orc.quant(orc.FMT_Q4_0, (0.05 * rng.standard_normal((n, k), dtype=np.float32)).astype(np.float32))
    act = rng.standard_normal((1, m, k), dtype=np.float32)
    act[0, m // 2] *= np.float32(1e36)
    got = ta.GgmlGemm().eval(ta.DeviceTensor.from_numpy(act), ta.Q40Weights(blocks, 1, n, k)).to_numpy().astype(np.float64)[0]
    wd = orc.dequant(orc.FMT_Q4_0, blocks, np.float32).reshape(n, k).astype(np.float64)
    want, size = act[0].astype(np.float64) @ wd.T, np.abs(act[0].astype(np.float64)) @ np.abs(wd).T
    # as in test_gpu_matvec.py: products are exact and at most k / 32 / 8 + 15 additions stand one after the other, each rounding by 2^-24 of a
    # partial sum that is no larger than the sum of the magnitudes; in f32 products round too and a block's are added one by one, k / 8 per wave
    steps = np.full((m, 1), k / 256 + 15)
    steps[m // 2 // 32 * 32 : m // 2 // 32 * 32 + 32] = k / 4 + 15   # (the rows that share blocks with the large one)
    assert np.all(np.abs(got - want) <= size * steps * 2.0 ** -24)


# f16 rows with k shared among waves: 32 x 16, 48 x 32, 64 x 32 and 32 x 64 (planes), 6 to 8 rows of tiles, and 16 x 64 of tall ones
@pytest.mark.parametrize("m,n,k", [(90, 1010, 1056), (290, 1010, 160), (290, 1001, 2080), (450, 1010, 1056), (470, 1001, 96), (150, 3001, 160), (149, 3000, 1056), (6, 4112, 1152), (7, 5136, 384), (8, 272, 2176), (8, 12240, 384), (9, 14352, 1152), (16, 16384, 256), (16, 8208, 128),
                                   # ... and those beside them that stay in one pass of the streaming kernel: all features in LDS, and four tiles a wave
                                   (6, 272, 12288), (7, 1040, 9216), (8, 528, 8192), (8, 4096, 4096), (6, 16, 4096)])
def test_shapes_with_k_shared_among_waves(rt, m, n, k):
    rng = np.random.default_rng(n + k + m)
    blocks = orc.quant(orc.FMT_Q4_0, (0.05 * rng.standard_normal((n, k), dtype=np.float32)).astype(np.float32))
    act = rng.standard_normal((1, m, k), dtype=np.float32).astype(np.float16)
    got = ta.GgmlGemm().eval(ta.DeviceTensor.from_numpy(act), ta.Q40Weights(blocks, 1, n, k)).to_numpy().astype(np.float64)[0]
    wd = orc.dequant(orc.FMT_Q4_0, blocks, np.float32).reshape(n, k).astype(np.float64)   # (not rounded to f16)
    want, size = act[0].astype(np.float64) @ wd.T, np.abs(act[0].astype(np.float64)) @ np.abs(wd).T
    # products are exact; at most k / 32 / 8 + 10 f32 additions stand one after the other, and the result is rounded to f16
    assert np.all(np.abs(got - want) <= size * (k / 256 + 11) * 2.0 ** -24 + np.abs(want) * 2.0 ** -11 + 2.0 ** -25)


# more activation rows than a grid has tiles of: the bits of the same rows in calls that fit (one pass over the weights in every case)
@pytest.mark.parametrize("m,n,k", [(65535 * 64 + 33, 33, 32), (65535 * 16 + 5, 16, 32), (65535 * 16 + 5, 16, 128)])
def test_more_f32_rows_than_a_grid_holds(rt, m, n, k):
    rng = np.random.default_rng(n)
    part = 999_936   # (whole tiles of every shape)
    blocks = orc.quant(orc.FMT_Q4_0, (0.05 * rng.standard_normal((n, k), dtype=np.float32)).astype(np.float32))
    w, op = ta.Q40Weights(blocks, 1, n, k), ta.GgmlGemm()
    act = rng.standard_normal((1, m, k), dtype=np.float32)
    got = op.eval(ta.DeviceTensor.from_numpy(act), w).to_numpy()[0]
    for at in range(0, m, part):
        want = op.eval(ta.DeviceTensor.from_numpy(np.ascontiguousarray(act[:, at : at + part])), w).to_numpy()[0]
        whole = min(part, m - at) // 64 * 64   # (the few rows left of a call may be given a tile of another shape)
        if whole > 512:
            np.testing.assert_array_equal(got[at : at + whole], want[:whole])
    tail = act[0, -40:].astype(np.float64) @ orc.dequant(orc.FMT_Q4_0, blocks, np.float32).reshape(n, k).astype(np.float64).T
    assert np.abs(got[-40:] - tail).max() <= 1e-5


# ... of several batches, over their own weights and over shared ones: planes and tiles
@pytest.mark.parametrize("batches,w_batches,n,k", [(2, 2, 16, 96), (2, 1, 16, 128), (4, 2, 15, 32)])
def test_more_f32_rows_than_a_grid_holds_in_batches(rt, batches, w_batches, n, k):
    rng = np.random.default_rng(n + batches)
    m = 65535 * 16 + 21
    blocks = [orc.quant(orc.FMT_Q4_0, (0.05 * rng.standard_normal((n, k), dtype=np.float32)).astype(np.float32)) for _ in range(w_batches)]
    act = np.zeros((batches, m, k), np.float32)
    rows = np.concatenate([[0, 1, 65535 * 16 - 1, 65535 * 16, m - 1], rng.integers(0, m, 30)])   # (the others are zeros)
    act[:, rows] = rng.standard_normal((batches, len(rows), k), dtype=np.float32)
    got = ta.GgmlGemm().eval(ta.DeviceTensor.from_numpy(act), ta.Q40Weights(np.concatenate([np.asarray(x).reshape(-1) for x in blocks]), w_batches, n, k)).to_numpy()
    for b in range(batches):
        w = orc.dequant(orc.FMT_Q4_0, blocks[b * w_batches // batches], np.float32).reshape(n, k).astype(np.float64)
        assert np.abs(got[b, rows] - act[b, rows].astype(np.float64) @ w.T).max() <= 1e-5
        assert np.count_nonzero(np.delete(got[b], rows, axis=0)) == 0
