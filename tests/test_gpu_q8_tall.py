"""f32 x Q8 on the 128 x 128 f16 tiles (q8_gemm.hip) at the edges of tiles, stages and blocks, against float64."""
import numpy as np
import pytest
import torch

from gpu_util import dev, host, say
from rumus_amd import nn

pytestmark = pytest.mark.gpu


# Rows: the fewest, a tile and one more, a last tile of 63.  Columns: fewer than a wave's 64, a tile and a few more.  K: one to
# five steps of 64 against a ring of three.  Blocks: two per step, one, three steps, all of K.  All below 1024 k, where
# these tiles are always taken.
@pytest.mark.parametrize("m,k,n,bs", [
    (65, 64, 36, 32), (65, 64, 36, 64), (128, 128, 128, 32), (129, 192, 132, 64), (191, 192, 260, 192), (256, 320, 200, 32),
    (257, 320, 130, 320), (300, 576, 300, 192), (511, 960, 129, 320), (1000, 256, 1024, 128), (2048, 512, 384, 256)])
def test_tall_tiles(m, k, n, bs):
    say(f"matmul_q8 128 x 128 tiles m={m} k={k} n={n} block {bs}")
    rng = np.random.default_rng(m + k + n + bs)
    x = (rng.normal(0, 1, (m, k)) * 10.0 ** rng.uniform(-6, 6, (m, 1))).astype(np.float32)
    x[:, rng.integers(0, k, 3)] *= 30.0
    x[3] = 0.0
    x[5, 7] = np.nan
    w = nn.quantize(dev(rng.normal(0, 0.02, (k, n)).astype(np.float32)), bs)
    got = host(nn.matmul(dev(x), w)).astype(np.float64)
    wd = host(nn.dequantize_kn(w)).astype(np.float64)
    rows = [r for r in range(m) if r != 5]
    exact = x[rows].astype(np.float64) @ wd
    terms = np.abs(x[rows]).astype(np.float64) @ np.abs(wd)
    # x as hi + lo: within 2^-22 of the element, or 2^-39 of the row's largest where lo is subnormal; a f32 sum of 2 k exact products and
    # k / bs scaled block sums, each addition within 2^-23 of what has been added up
    top = np.abs(x[rows]).max(axis=1, keepdims=True) * np.abs(wd).sum(axis=0, keepdims=True)
    bound = terms * (2 * k + 2 * (k // bs) + 8) * 2.0 ** -23 + top * 2.0 ** -39
    assert np.isnan(got[5]).all()
    assert (np.abs(got[rows] - exact) <= bound).all()
    # an ordinary sum's error grows like the root of its length: a misplaced element shows here
    err = np.linalg.norm(got[rows] - exact, axis=1) / (np.linalg.norm(exact, axis=1) + 1e-300)
    assert np.delete(err, 3).max() < 1e-5
