"""grad_x of larger batches (w4t_wide_kernel) where its split begins and ends: against the narrow kernel's operation and float64."""
import numpy as np
import pytest

import oracle
from gpu_util import dev, host, say

pytestmark = pytest.mark.gpu


def takes_the_matrix_cores(m, k, n, g):
    """Whether the call wants workspace, which the vector kernel does not: asked for on a stream that has none and is being captured."""
    import torch
    from rumus_amd import ops
    words = torch.zeros((k // 8, n), dtype=torch.int32, device="cuda")
    meta = torch.ones((-(-k // g), n), dtype=torch.float32, device="cuda")
    gy, out = torch.zeros((m, n), device="cuda"), torch.empty((m, k), device="cuda")
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        out.zero_()
        try:
            ops.qmatmul_int4_t(gy, words, meta, meta, k, g, out=out)
        except ops.RumusError as e:
            assert "workspace of" in str(e)
            return True
    return False


# n: one step of 16 (three of a workgroup's waves have none), two, five, six; 8 and 9 steps a wave in one share, shares of a few steps;
# m: one row past the smallest batch, a tile of 64, one over it, several; k: part of a tile of 128, groups of 128 and 256
@pytest.mark.parametrize("n", [16, 32, 80, 96, 512, 560, 2064])
@pytest.mark.parametrize("m,k,g", [(33, 256, 128), (64, 128, 128), (65, 388, 128), (200, 512, 256), (129, 1500, 128),
                                   # the first three, with weights that the vector kernel does not take
                                   (33, 3072, 128), (64, 2048, 128), (65, 1924, 128)])
def test_grad_x_wide(m, k, n, g):
    from rumus_amd import ops
    say(f"qmatmul_int4_t wide m={m} k={k} n={n} g={g}")
    rng = np.random.default_rng(m * 7 + n)
    w = rng.normal(0, 0.02, (k, n)).astype(np.float32)
    w[:, 1::5] += 0.3                                        # zero-points far outside 0 .. 15
    gy = (rng.normal(0, 1, (m, n)) * 10.0 ** rng.uniform(-6, 6, (m, 1))).astype(np.float32)
    gy[2] = 0.0
    gy[4, n - 1] = np.inf                                    # in the last column: its own row only
    gy[m - 1, 0] = np.nan
    packed, scales, zp = oracle.w4_from_f32(w, g)
    got = host(ops.qmatmul_int4_t(dev(gy), dev(packed), dev(scales), dev(zp), k, g)).astype(np.float64)
    deq = oracle.w4_dequant(packed, scales, zp, k, g).astype(np.float64)
    rows = [r for r in range(m) if r not in (2, 4, m - 1)]
    exact = gy[rows].astype(np.float64) @ deq.T
    # the bound of test_gpu_w4_t_steps.py: each factor pair rounded once in f32 and cut to 2^-21 by the hi and lo halves, 2 n additions in
    # f32 of magnitudes up to (|q - z0| + |zp - z0|) scales
    reach = (15.5 + np.abs(zp - np.rint(zp)) + np.maximum(np.abs(zp) - 15.0, 0.0)) * scales
    size = np.abs(gy[rows]).astype(np.float64) @ np.repeat(reach, g, axis=0)[:k].astype(np.float64).T
    assert (np.abs(got[rows] - exact) <= size * (2.0 ** -20 + 2 * n * 2.0 ** -23)).all()
    # and an ordinary sum's error stays far below that: a misplaced element or a step added twice shows here
    err = np.linalg.norm(got[rows] - exact, axis=1) / np.linalg.norm(exact, axis=1)
    assert err.max() < 2e-5
    assert not got[2].any()
    assert not np.isfinite(got[4]).any() and not np.isfinite(got[m - 1]).any()


# few columns: the last three weights of the test above at each of its n, and one of 512 tiles and more
@pytest.mark.parametrize("m,k,n", [(m, k, n) for n in (16, 32, 80, 96, 512, 560, 2064) for m, k in ((33, 3072), (64, 2048), (65, 1920))] +
                         [(512, 4096, 112), (256, 11008, 112), (384, 11008, 112)])
def test_few_columns_take_the_matrix_cores(m, k, n):
    say(f"qmatmul_int4_t route m={m} k={k} n={n}")
    assert takes_the_matrix_cores(m, k, n, 128)


def test_few_columns_of_many_tiles():
    test_grad_x_wide(384, 11008, 112, 128)
