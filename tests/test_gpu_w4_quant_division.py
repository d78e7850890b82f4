"""The INT4 quantizers' division by a group's scale (w4_quant.hip), bit for bit against the CPU oracle, where it can go wrong: both
sides of the range that the short division is held to, elements that sit on the ties of the rounding, and tiny elements."""
import numpy as np
import pytest

import oracle
from gpu_util import dev, host, host_u32, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("g", [8, 32, 64, 128])
@pytest.mark.parametrize("kind", ["magnitudes", "ties", "tiny", "edges"])
def test_quantize_pack_division(g, kind):
    from rumus_amd import ops
    say(f"w4 quantizers, division, {kind} g={g}")
    rng = np.random.default_rng(g)
    k, n = 4 * g, 1024
    w = rng.normal(0, 1, (k, n))
    if kind == "magnitudes":                                 # scales from 2^-80 to 2^80
        w = w * 2.0 ** np.linspace(-80, 80, n)
    elif kind == "ties":                                     # quotients on and an ulp beside k + 1/2, at scales of every mantissa
        step = rng.uniform(0.001, 0.002, n).astype(np.float32)
        w = ((rng.integers(0, 31, (k, n)) / 2.0).astype(np.float32) * step).astype(np.float32)
        w[::g], w[1::g] = 0.0, 15.0 * step
        w = (w.view(np.int32) + rng.integers(-1, 2, w.shape) * (w > 0)).view(np.float32)
    elif kind == "tiny":                                     # elements far below the scale, down to subnormals
        w = w * 10.0 ** rng.uniform(-44, 0, (k, n))
    else:                                                    # scales within a few ulp of 2^-60 and 2^60
        w = np.clip(w, -2, 2) * 2.0 ** np.where(np.arange(n) % 2, 58.0, -57.0) * (1 + rng.integers(-3, 4, n) * 2.0 ** -23)
        w[::g], w[1::g] = 7.5 * 2.0 ** np.where(np.arange(n) % 2, 57.0, -60.0), -7.5 * 2.0 ** np.where(np.arange(n) % 2, 57.0, -60.0)
    w = np.ascontiguousarray(w, np.float32)
    for sym in (False, True):
        want = oracle.w4_from_f32(w, g, symmetric=sym)
        got = ops.w4_quantize_pack(dev(w), g, sym)
        np.testing.assert_array_equal(host_u32(got[0]), want[0])
        np.testing.assert_array_equal(host(got[1]), want[1])
        np.testing.assert_array_equal(host(got[2]), want[2])
    want = oracle.w4_awq_from_f32(w, g)
    got = ops.w4_quantize_pack_awq(dev(w), g)
    np.testing.assert_array_equal(host_u32(got[0]), want[0])
    np.testing.assert_array_equal(host(got[1]), want[1])
    np.testing.assert_array_equal(host_u32(got[2]), want[2])
