"""f16 activations through the integer matrix-core kernel (w4_gemm_i8.hip reads and writes f16 itself there): bit for bit what the
f32 call gives, rounded once, over the forms that the route accepts and refuses."""
import numpy as np
import pytest
import torch

import oracle
from gpu_util import dev, host, say

pytestmark = pytest.mark.gpu


# m: each height of a workgroup, whole and ragged row tiles.  k: multiples of 8, of 4 and of neither (the last inside a padded
# group), shares beyond the registers' 2048.  n: one to four columns per lane, ragged last tiles.  offset: elements that x and y begin
# behind an aligned address (4: 8 bytes, taken directly; 1: through f32 copies).
@pytest.mark.parametrize("m,k,n,g", [(9, 256, 64, 64), (16, 2000, 1000, 64), (33, 1004, 260, 128), (47, 1003, 516, 128), (65, 516, 4100, 64),
                                     (100, 2048, 11008, 128), (128, 520, 36, 64), (300, 4096, 4096, 128), (17, 17408, 132, 128)])
@pytest.mark.parametrize("offset", [0, 4, 1])
def test_f16_direct(m, k, n, g, offset):
    from rumus_amd import ops
    say(f"qmatmul_int4_f16 m={m} k={k} n={n} g={g} offset {offset}")
    rng = np.random.default_rng(m + k + n)
    packed, scales, zp = (dev(a) for a in oracle.w4_from_f32(rng.normal(0, 0.02, (k, n)).astype(np.float32), g))
    x16 = (rng.normal(0, 1, (m, k)) * 10.0 ** rng.uniform(-4, 2, (m, 1))).astype(np.float16)
    x16[1] = 0.0
    x16[2, k - 1] = np.inf
    x16[3] = 60000.0                                          # results beyond the range of f16
    bias = dev(rng.normal(0, 0.01, n).astype(np.float32))
    x = torch.zeros(m * k + offset, dtype=torch.float16, device="cuda")[offset:].view(m, k).copy_(dev(x16))
    y = torch.full((m * n + offset + 8,), 7.0, dtype=torch.float16, device="cuda")
    out = y[offset:offset + m * n].view(m, n)
    ops.qmatmul_int4_f16(x, packed, scales, zp, k, g, bias=bias, out=out)
    want = host(ops.qmatmul_int4(x.float(), packed, scales, zp, k, g, bias=bias))
    with np.errstate(over="ignore"):
        np.testing.assert_array_equal(host(out), want.astype(np.float16))
    assert bool((y[:offset] == 7.0).all()) and bool((y[offset + m * n:] == 7.0).all())
