"""f32 x Q8, small batches whose K is shared over workgroups (q8_gemm.hip), and K shorter than the ring of stages, against float64."""
import numpy as np
import pytest

from gpu_util import dev, host, say

pytestmark = pytest.mark.gpu


# 18 steps of 64 k in three shares, 30 in six, 32 in six with two left for the last; blocks of 96: periods of three halves of a step, 45
# steps in eight shares with three for the last, 40.5 in seven; periods of two, four and sixteen steps; one share where the
# tiles fill the chip; K of one, two and three steps against a ring of three; more than 32 rows
@pytest.mark.parametrize("m,k,n,bs", [
    (5, 1152, 100, 32), (13, 1152, 9632, 32), (30, 2048, 2048, 32), (32, 2080, 130, 32), (32, 1920, 260, 64), (17, 2880, 300, 96),
    (32, 2592, 128, 96), (9, 4096, 1000, 128), (24, 3072, 520, 1024), (6, 4096, 640, 4096), (16, 1152, 33000, 32), (32, 64, 100, 32),
    (5, 128, 36, 64), (7, 192, 132, 32), (31, 96, 132, 96), (40, 2592, 256, 96), (64, 1152, 300, 32), (70, 2880, 130, 96),
    # one block per column beyond 64 rows: K is cut inside it, in periods of 32, 4, 2, 11, 31, 13 and 1 halves of a step
    (70, 2048, 130, 2048), (66, 5248, 200, 5248), (250, 2752, 100, 2752), (100, 1056, 70, 1056), (66, 992, 64, 992), (130, 2080, 300, 2080),
    (65, 1696, 40, 1696), (300, 4096, 1000, 2048)])
def test_shares_of_k(m, k, n, bs):
    from rumus_amd import nn
    say(f"matmul_q8 m={m} k={k} n={n} block {bs}")
    rng = np.random.default_rng(m + k + n + bs)
    x = (rng.normal(0, 1, (m, k)) * 10.0 ** rng.uniform(-6, 6, (m, 1))).astype(np.float32)
    x[3] = 0.0
    x[4, k - 1] = np.nan
    w = nn.quantize(dev(rng.normal(0, 0.02, (k, n)).astype(np.float32)), bs)
    got = host(nn.matmul(dev(x), w)).astype(np.float64)
    wd = host(nn.dequantize_kn(w)).astype(np.float64)
    rows = [r for r in range(m) if r != 4]
    exact = x[rows].astype(np.float64) @ wd
    terms = np.abs(x[rows]).astype(np.float64) @ np.abs(wd)
    # x within 2^-22 of an element in two halves, 2^-27 of the row's largest in four digits; f32 sums of 2 k products and k / bs scaled block
    # sums, each addition within 2^-23 of what has been added up
    top = np.abs(x[rows]).max(axis=1, keepdims=True) * np.abs(wd).sum(axis=0, keepdims=True)
    bound = terms * (2 * k + 2 * (k // bs) + 8) * 2.0 ** -23 + top * 2.0 ** -27
    assert np.isnan(got[4]).all()
    assert (np.abs(got[rows] - exact) <= bound).all()
    # an ordinary sum's error grows like the root of its length: a step left out, or added twice, shows here
    err = np.linalg.norm(got[rows] - exact, axis=1) / (np.linalg.norm(exact, axis=1) + 1e-300)
    assert np.delete(err, 3).max() < 1e-5
