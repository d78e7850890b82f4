"""INT4 forward for 2 to 8 rows on the int8 matrix cores (``w4_gemv_mfma.hip``): units of 128 and 256 k and their tails, groups of 32, 64 and
128, column tiles, act-order rows in one launch and in parts, f16 rows, elements far apart in a unit, NaN and infinity.

The bound, against float64: an activation is rounded to 2^-22 of its unit's largest magnitude (2^-21 where that lies within 1.6 % below a power of
two), so an output is off by at most max|x| 2^-21 sum|w|, half of what ``check`` allows; the f32 sums around it lose less than 2^-20 of the
summed magnitudes (up to K/128 + 8 additions of 2^-24 each)."""
import numpy as np
import pytest

from gpu_util import dev, host, say

import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from rumus_amd import ops
    return ops


def weights(rng, k, n, g, zero="float"):
    packed, scales, zp = oracle.w4_from_f32(rng.normal(0, 0.02, (k, n)).astype(np.float32), g)
    if zero == "integer":
        zp = np.clip(np.rint(zp), 0, 15).astype(np.float32)
    q = oracle.w4_unpack(packed, packed.shape[0] * 8).astype(np.float64)[:k]
    rows = np.arange(k) // g
    return packed, scales, zp, (q - zp[rows].astype(np.float64)) * scales[rows].astype(np.float64)


def check(got, x, w, largest=None):
    x = x.astype(np.float64)
    want = x @ w
    top = np.abs(x).max(axis=1, keepdims=True) if largest is None else largest
    bound = 2.0 ** -20 * (top * np.abs(w).sum(axis=0) + np.abs(x) @ np.abs(w))
    worst = float((np.abs(got - want) / bound).max())
    assert worst <= 1.0, worst


SHAPES = [(2, 32, 16, 32), (3, 96, 20, 32), (8, 160, 48, 32), (2, 1000, 52, 64), (5, 1088, 64, 64), (4, 128, 4, 128), (7, 1152, 36, 128),
          (2, 2048, 80, 128), (6, 2176, 16, 128), (3, 4096, 64, 256), (8, 4224, 32, 128), (4, 8320, 32, 64), (4, 512, 8192, 128),
          (8, 300, 8224, 32), (3, 1001, 16, 8 * 32),
          # groups of 32 on more workgroups than compute units; eight rows on two of them; wide row-major weights of groups of 64
          (5, 1088, 4112, 32), (3, 2176, 4128, 32), (7, 2176, 4128, 128), (3, 2176, 12288, 64)]


@pytest.mark.parametrize("m,k,n,g", SHAPES)
@pytest.mark.parametrize("tiled", [False, True])
def test_few_rows_against_float64(ops, m, k, n, g, tiled):
    if tiled and n % 16:
        pytest.skip("the decode layout wants whole tiles")
    say(f"few rows m={m} k={k} n={n} g={g} tiled={tiled}")
    rng = np.random.default_rng(m * 7 + k + n)
    packed, scales, zp, w = weights(rng, k, n, g)
    x = rng.normal(0, 1, (m, k)).astype(np.float32)
    d = [dev(a) for a in (packed, scales, zp)]
    if tiled:
        got = host(ops.qmatmul_int4_decode(dev(x), *ops.w4_decode_layout(*d, g), k, g))
    else:
        got = host(ops.qmatmul_int4(dev(x), *d, k, g))
    check(got, x, w)
    if not tiled and k % 4 == 0:             # a row does not depend on the others
        one = host(ops.qmatmul_int4(dev(np.ascontiguousarray(np.concatenate([x[-1:], x[:1] * 3, x[:1]]))), *d, k, g))
        if k <= 2048 or m > 2:
            np.testing.assert_array_equal(one[0], got[-1])
    if not tiled and k % 8 == 0:             # f16 rows: the same kernel, rounded once
        xh = x.astype(np.float16)
        f32 = host(ops.qmatmul_int4(dev(xh.astype(np.float32)), *d, k, g))
        np.testing.assert_array_equal(host(ops.qmatmul_int4_f16(dev(xh), *d, k, g)), f32.astype(np.float16))


@pytest.mark.parametrize("m,k", [(2, 256), (8, 2048), (4, 4096), (8, 4096), (3, 8192), (5, 12288), (2, 16384), (2, 32768),
                                 (4, 6144), (4, 6272), (3, 8320), (2, 12288), (2, 12416)])
def test_act_order_rows_in_parts(ops, m, k):
    n, g = 48, 128
    say(f"few rows act-order m={m} k={k}")
    rng = np.random.default_rng(m + k)
    packed, scales, zp, w = weights(rng, k, n, g)
    perm = rng.permutation(k).astype(np.int32)
    x = rng.normal(0, 1, (m, k)).astype(np.float32)
    t = ops.w4_decode_layout(dev(packed), dev(scales), dev(zp), g)
    got = host(ops.qmatmul_int4_decode(dev(x), *t, k, g, perm=dev(perm)))
    check(got, x[:, perm], w)


@pytest.mark.parametrize("m,k,g", [(3, 256, 128), (4, 1000, 64), (8, 4096, 128), (2, 992, 32)])
@pytest.mark.parametrize("power", [7, 9, 20, 60])
def test_elements_far_apart(ops, m, k, g, power):
    """Channels 2^power as large that meet weights of zero: what the others add up to keeps its bits."""
    say(f"few rows far apart m={m} k={k} g={g} power={power}")
    n = 32
    rng = np.random.default_rng(power + k)
    packed, scales, zp, w = weights(rng, k, n, g, zero="integer")
    loud = rng.permutation(k)[:max(1, k // 64)]
    for c in loud:                                          # code = zero-point: a weight of zero
        z = zp[c // g].astype(np.uint32)
        shift = np.uint32(4 * (c % 8))
        packed[c // 8] = (packed[c // 8] & ~(np.uint32(15) << shift)) | (z << shift)
        w[c] = 0.0
    x = rng.normal(0, 1, (m, k)).astype(np.float32)
    x[1, loud] *= np.float32(2.0 ** power)                  # one row: its neighbours stay as they are
    got = host(ops.qmatmul_int4(dev(x), dev(packed), dev(scales), dev(zp), k, g))
    # up to 2^8 apart the plain bound; beyond, every element counts with its own bits and only sums round
    largest = np.abs(x).max(axis=1, keepdims=True).astype(np.float64)
    largest[1] = min(largest[1], 2.0 ** 10)
    y = x.copy()
    y[1, loud] = 0.0
    check(got, y, w, largest)


def test_not_finite_and_tiny(ops):
    m, k, n, g = 4, 1024, 32, 128
    rng = np.random.default_rng(5)
    packed, scales, zp, w = weights(rng, k, n, g)
    x = rng.normal(0, 1, (m, k)).astype(np.float32)
    x[1, 77] = np.nan
    x[2, 1000] = -np.inf
    x[3] *= np.float32(2.0 ** -100)
    got = host(ops.qmatmul_int4(dev(x), dev(packed), dev(scales), dev(zp), k, g))
    assert not np.isfinite(got[1:3]).any()
    check(got[[0, 3]], x[[0, 3]], w)


# K of which the last sweep leaves units without elements, and a unit that ends inside a step of 64: every array the last thing in its
# memory but for NaNs, which none of those may read
@pytest.mark.parametrize("m,k,n,g", [(4, 4224, 12288, 128), (8, 2304, 8192, 128), (3, 1056, 48, 32), (6, 4192, 64, 32)])
@pytest.mark.parametrize("form", ["plain", "tiled", "zp4", "act", "half", "norm", "glu"])
def test_units_past_the_end(ops, m, k, n, g, form):
    import torch
    say(f"few rows, units past the end m={m} k={k} n={n} g={g} {form}")
    gen = torch.Generator(device="cuda").manual_seed(m + k + n)

    def last(t):
        room = torch.full((t.numel() + 4096,), float("nan") if t.is_floating_point() else 0x7FC00000, dtype=t.dtype, device="cuda")
        room[:t.numel()] = t.reshape(-1)
        return room[:t.numel()].view(t.shape)

    packed = torch.randint(-2 ** 31, 2 ** 31 - 1, (k // 8, n), generator=gen, device="cuda", dtype=torch.int32)
    scales = 0.01 + 0.01 * torch.rand((k // g, n), generator=gen, device="cuda")
    zp = torch.randint(0, 16, (k // g, n), generator=gen, device="cuda").float()
    x = torch.randn((m, k), generator=gen, device="cuda")
    perm = torch.randperm(k, generator=gen, device="cuda")
    q = torch.stack([(packed >> (4 * i)) & 15 for i in range(8)], 1).reshape(k, n).double()
    w = (q - zp.double().repeat_interleave(g, 0)) * scales.double().repeat_interleave(g, 0)
    d = [last(t) for t in (packed, scales, zp)]
    tiled = [last(t) for t in ops.w4_decode_layout(*d, g)]
    if form == "plain":
        got = ops.qmatmul_int4(last(x), *d, k, g)
    elif form == "tiled":
        got = ops.qmatmul_int4_decode(last(x), *tiled, k, g)
    elif form == "zp4":
        z4 = zp.to(torch.int64).view(k // g, n // 8, 8)
        z4 = sum(z4[..., i] << (4 * i) for i in range(8))
        got = ops.qmatmul_int4_zp4(last(x), d[0], d[1], last(torch.where(z4 >= 2 ** 31, z4 - 2 ** 32, z4).to(torch.int32)), k, g)
    elif form == "act":
        got = ops.qmatmul_int4_decode(last(x), *tiled, k, g, perm=last(perm.to(torch.int32)))
        x = x[:, perm]
    elif form == "half":
        x = x.half()
        got = ops.qmatmul_int4_f16(last(x), *d, k, g).float()
    elif form == "norm":
        scale = 1.0 + 0.1 * torch.randn(k, generator=gen, device="cuda")
        got = ops.qmatmul_int4_decode_block(last(x), *tiled, k, g, norm_weight=last(scale), eps=1e-6)
        x = x.double() * scale.double() / (x.double().square().mean(1, keepdim=True) + 1e-6).sqrt()
    else:
        up = torch.randn((m, k), generator=gen, device="cuda")
        got = ops.qmatmul_int4_decode_block(last(torch.cat([x, up], 1)), *tiled, k, g, swiglu=True)
        x = x.double() * torch.sigmoid(x.double()) * up.double()
    want = x.double() @ w
    # activations within 2^-20 of their unit's largest, f32 around them; one rounding to f16
    bound = (2.0 ** -11 if form == "half" else 2.0 ** -18) * (x.double().abs() @ w.abs() + x.double().abs().amax(1, keepdim=True) * w.abs().sum(0))
    assert float(((got.double() - want).abs() / bound).max()) <= 1.0


# Activations of 22 bits, odd multiples of 2^-21 below 1.96, of which a column adds up four: 24 bits, nothing is rounded.  With activations cut
# to 21 bits every one of them would be off by 2^-22.
@pytest.mark.parametrize("m,k,n,g,form", [
    (2, 512, 32, 128, "plain"), (2, 2048, 48, 64, "tiled"), (3, 4224, 36, 128, "plain"), (4, 1024, 20, 32, "plain"), (8, 4096, 4096, 128, "tiled"),
    (5, 2304, 8224, 128, "plain"), (4, 4096, 11008, 128, "plain"), (3, 1001, 16, 256, "plain"), (6, 2048, 64, 128, "act"), (4, 4096, 48, 64, "act"),
    # two rows of a weight that is read for longer than the rows are converted
    (2, 16384, 9616, 128, "plain")])
def test_bits_of_the_activations(ops, m, k, n, g, form):
    say(f"few rows, 22 bits m={m} k={k} n={n} g={g} {form}")
    rng = np.random.default_rng(m + k + n)
    words = -(-k // g) * g // 8
    at = np.stack([rng.choice(k, 4, replace=False) for _ in range(n)], 1)        # a column's four weights of one
    packed = np.zeros((words, n), np.uint32)
    np.bitwise_or.at(packed, (at // 8, np.arange(n)), np.uint32(1) << (4 * (at % 8)).astype(np.uint32))
    scales, zp = np.ones((words * 8 // g, n), np.float32), np.zeros((words * 8 // g, n), np.float32)
    d = [dev(a) for a in (packed, scales, zp)]
    x = ((4.0 * rng.integers(-2 ** 18, 2 ** 18, (m, k)) + 1.0) * 2.0 ** -21).astype(np.float32)
    large = x[:, ::64].shape
    x[:, ::64] = (4.0 * rng.integers(2 ** 19, int(1.96 * 2 ** 19), large) + 1.0) * 2.0 ** -21 * rng.choice([-1.0, 1.0], large)
    perm = rng.permutation(k) if form == "act" else np.arange(k)
    if form == "plain":
        got = host(ops.qmatmul_int4(dev(x), *d, k, g))
    else:
        got = host(ops.qmatmul_int4_decode(dev(x), *ops.w4_decode_layout(*d, g), k, g, perm=dev(perm.astype(np.int32)) if form == "act" else None))
    np.testing.assert_array_equal(got, x[:, perm].astype(np.float64)[:, at].sum(axis=1))


@pytest.mark.parametrize("m,k,g", [(8, 256, 128), (4, 1024, 64), (8, 2304, 128), (7, 512, 32)])
@pytest.mark.parametrize("large", [240.0, 700.0, 1000.0])
def test_elements_far_apart_and_zero_points_far_away(ops, m, k, g, large):
    """Rows of one value and a few tiny ones, zero-points of several hundred: the digits' sums times the zero-points."""
    say(f"few rows far apart m={m} k={k} g={g}, zero-points up to {large}")
    n = 32
    rng = np.random.default_rng(m + k)
    packed, scales, zp, _ = weights(rng, k, n, g)
    zp = (large * rng.uniform(0.9, 1.0, zp.shape) * rng.choice([-1.0, 1.0], zp.shape)).astype(np.float32)
    q = oracle.w4_unpack(packed, packed.shape[0] * 8).astype(np.float64)[:k]
    rows = np.arange(k) // g
    w = (q - zp[rows].astype(np.float64)) * scales[rows].astype(np.float64)
    x = np.repeat(np.linspace(1.0, 1.95, m * 16).astype(np.float32).reshape(16, m, 1), k, axis=2)
    x[:, :, np.arange(k) % 64 < 8] *= np.float32(2.0 ** -12)     # all elements of some lanes: every unit is multiplied in parts then
    d = [dev(a) for a in (packed, scales, zp)]
    for rows_of in x:
        got = host(ops.qmatmul_int4(dev(rows_of), *d, k, g))
        check(got, rows_of, w)
