"""grad_x on the matrix cores (w4_gemm_t.hip) where its pipeline over n begins and ends: fewer steps than slots, shares of n that
end inside a call's columns, remainders of a step, each width of a workgroup; against float64."""
import numpy as np
import pytest

import oracle
from gpu_util import dev, host, say

pytestmark = pytest.mark.gpu


# n: one step of 32 (whole and ragged), two, three, four; 36 steps in two shares, 67 in four, the last share the shorter
# one; 128 rows and more at few columns: several shares of many row tiles.  m: half a tile of 64, one over it, a whole one, one more.
@pytest.mark.parametrize("n", [4, 32, 36, 64, 92, 96, 128, 1148, 2116])
@pytest.mark.parametrize("m,k,g", [(32, 256, 128), (33, 128, 128), (64, 192, 64), (129, 256, 128), (49, 96, 32), (25, 128, 64),
                                   # weights too large for the vector kernel: one step a share, several, shares that end in a short one
                                   (32, 4096, 128), (33, 3072, 128), (64, 1536, 64), (129, 1024, 128), (49, 2048, 32), (25, 4096, 64), (300, 512, 32)])
def test_grad_x_steps(m, k, n, g):
    from rumus_amd import ops
    say(f"qmatmul_int4_t steps m={m} k={k} n={n} g={g}")
    rng = np.random.default_rng(m * 7 + n)
    w = rng.normal(0, 0.02, (k, n)).astype(np.float32)
    gy = (rng.normal(0, 1, (m, n)) * 10.0 ** rng.uniform(-6, 6, (m, 1))).astype(np.float32)
    gy[2] = 0.0
    gy[4, n - 1] = np.inf                                    # in the last column: its own row only
    packed, scales, zp = oracle.w4_from_f32(w, g)
    got = host(ops.qmatmul_int4_t(dev(gy), dev(packed), dev(scales), dev(zp), k, g)).astype(np.float64)
    deq = oracle.w4_dequant(packed, scales, zp, k, g).astype(np.float64)
    rows = [r for r in range(m) if r not in (2, 4)]
    exact = gy[rows].astype(np.float64) @ deq.T
    # a term is grad_y scale (q - z0) less grad_y scale (zp - z0), each factor pair rounded once in f32 and cut to 2^-21 by the hi and lo halves;
    # 2 n additions in f32, each within 2^-23 of the magnitudes added up (|q - z0| <= 15.5 scales)
    s_big = np.repeat(scales.reshape(-1, n), g, axis=0)[:k].astype(np.float64)
    size = np.abs(gy[rows]).astype(np.float64) @ (15.5 * s_big).T
    assert (np.abs(got[rows] - exact) <= size * (2.0 ** -20 + 2 * n * 2.0 ** -23)).all()
    # and an ordinary sum's error stays far below that: a misplaced element or a step added twice shows here
    err = np.linalg.norm(got[rows] - exact, axis=1) / np.linalg.norm(exact, axis=1)
    assert err.max() < 2e-5
    assert not got[2].any()
    assert not np.isfinite(got[4]).any()
