"""W4 forward on the six-bit-float matrix cores (large batches; qmatmul_int4.wgsl:40-87) at the edges of its tiles, against
the float64 product."""
import numpy as np
import pytest
import torch

import oracle
from gpu_util import dev, host, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from rumus_amd import ops as o
    return o


# All of these are taken by that kernel.  Rows: blocks of 128 (last one of 1, 77 or 60 rows, or full); columns: tiles of
# 256 (first two), 384 and 512, with a right edge inside a lane's columns or none; K: an even and an odd number of steps of
# 64, padded (1500 -> 1536, 1028 and 1090 -> 1152) or not.
@pytest.mark.parametrize("m,k,n,g,act_order,zeros", [
    (1409, 1500, 2820, 64, False, "fractional"), (1408, 1024, 2816, 128, True, "integer"),
    (1100, 1024, 6144, 128, True, "u4"), (1357, 1090, 6148, 64, False, "fractional"), (1400, 1152, 6144, 192, True, "fractional"),
    (3516, 1028, 4100, 128, False, "fractional"), (3500, 1088, 4096, 64, True, "u4"), (3584, 1024, 4096, 256, False, "integer")])
def test_six_bit_kernel_at_its_edges(ops, m, k, n, g, act_order, zeros):
    say(f"w4 forward, six-bit kernel m={m} k={k} n={n} g={g} act_order={act_order} zero-points {zeros}")
    if zeros != "u4":                          # (asked for whole words of eight k)
        assert ops.qmatmul_int4_block_takes(m, k // 8 * 8, n, g)
    rng = np.random.default_rng(m + k + n)
    padded = -(-k // g) * g
    w = rng.normal(0, 0.02, (k, n)).astype(np.float32)
    packed, scales, zp = oracle.w4_from_f32(w, g)
    if zeros != "fractional":
        zp = np.clip(np.rint(zp), 0, 15).astype(np.float32)
    scales[0, 3] = 0.0
    x = rng.normal(0, 1, (m, k)).astype(np.float32)
    x *= (10.0 ** rng.uniform(-12, 12, (m, 1))).astype(np.float32)
    # elements that tower over their neighbours; one of them, 2^18 larger, meets weights of exactly zero where zero-points are
    # integers: what is left of those rows is their small elements
    perm_np = rng.permutation(k).astype(np.int32) if act_order else np.arange(k, dtype=np.int32)
    x[5:9, perm_np[700]] *= 1000.0
    x[m - 1, perm_np[k - 1]] *= 3000.0
    if zeros != "fractional":
        z = zp[40 // g].astype(np.uint32)
        packed[40 // 8] = (packed[40 // 8] & ~np.uint32(15)) | z
        x[7:11, perm_np[40]] *= np.float32(2.0 ** 18)
    x[2, 9] = np.inf
    bias = np.zeros(n, np.float32)
    d = [dev(packed), dev(scales)]
    if zeros == "u4":
        q = np.rint(zp).astype(np.uint32).reshape(zp.shape[0], n // 8, 8)
        qzeros = (q << (4 * np.arange(8, dtype=np.uint32))).sum(axis=2, dtype=np.uint32).view(np.int32)
        got = host(ops.qmatmul_int4_zp4(dev(x), *d, dev(qzeros), k, g, bias=dev(bias), perm=dev(perm_np) if act_order else None))
    elif act_order:
        got = host(ops.qmatmul_int4_perm(dev(x), *d, dev(zp), k, g, bias=dev(bias), perm=dev(perm_np)))
    else:
        got = host(ops.qmatmul_int4(dev(x), *d, dev(zp), k, g, bias=dev(bias)))
    assert np.isnan(got[2]).all()
    rows = np.r_[0:2, 3:40, 120:140, m // 2:m // 2 + 30, m - 40:m]
    xs = x[rows][:, perm_np].astype(np.float64)
    groups = np.repeat(np.arange(scales.shape[0]), g)[:k]
    q = oracle.w4_unpack(packed, k).astype(np.float64)
    z = np.clip(np.rint(zp), 0, 15)[groups].astype(np.float64)
    rest = zp[groups] - z
    s = scales[groups].astype(np.float64)
    exact = xs @ ((q - z - rest) * s)
    terms = np.abs(xs) @ ((np.abs(q - z) + np.abs(rest)) * np.abs(s))
    # sums: six additions and one change of scale per step of 64, 7 2^-24 of what has been added up, two additions per group for the
    # zero-points' rest, each within 2^-23 of that; values within 2^-29 of the largest of 32 (2^-39 where one of them towers), under
    # 4 2^-23 of ordinary terms, and their bf16 thirds in the rest's products another 2^-23
    steps = padded // 64
    bound = (6 * steps + 2 * scales.shape[0] + 8) * 2.0 ** -23
    err = np.abs(got[rows] - exact) / (terms + 1e-300)
    say(f"    worst error / bound {err.max() / bound:.3f}")
    assert (err <= bound).all()


# Long rows, where the preparation takes two rows or one per workgroup, and groups that pad K beyond what it takes (then
# another kernel runs).  The stream's workspace holds another call's digits, exponents and sums, every run of 32 marked
# there, and the padding nibbles are 15: what a kernel reads without having written it shows.  (At k = 5120 the rows go in two halves
# where the workspace cannot grow: test_gpu_workspace_room.py.)
@pytest.mark.parametrize("k,g,taken", [(4096, 128, True), (5120, 128, True), (7000, 192, True), (11008, 64, True), (16384, 128, True), (16320, 192, True),
                                       (16384, 192, False), (16384, 384, False), (16136, 384, False), (14336, 6144, False), (9224, 9216, False)])
def test_long_rows(ops, k, g, taken):
    m, n = 1500, 4096
    say(f"w4 forward m={m} k={k} n={n} g={g}, six-bit kernel: {taken}")
    assert ops.qmatmul_int4_block_takes(m, k, n, g) == taken
    gen = torch.Generator(device="cuda").manual_seed(k + g)
    normal = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    packed, scales, zp = ops.w4_quantize_pack(normal(k, n) * 0.02, g)
    other = normal(2000, 4096)
    other[:, ::32] *= 1e5
    ops.qmatmul_int4(other, *ops.w4_quantize_pack(normal(4096, n) * 0.02, 64), 4096, 64)
    packed[k // 8:] = -1
    x = normal(m, k)
    x[5:9, k - 30] *= 1000.0
    x[m - 1, 100] *= 3000.0
    got = ops.qmatmul_int4(x, packed, scales, zp, k, g)
    rows = torch.cat([torch.arange(40), torch.arange(700, 740), torch.arange(m - 40, m)]).cuda()
    q = torch.stack([(packed[:k // 8] >> (4 * i)) & 15 for i in range(8)], 1).reshape(k, n).double()
    expand = lambda t: t.double().repeat_interleave(g, 0)[:k]
    z, s, xs = expand(zp), expand(scales), x[rows].double()
    exact = xs @ ((q - z) * s)
    near = z.round().clamp(0, 15)
    terms = xs.abs() @ (((q - near).abs() + (z - near).abs()) * s.abs())
    padded, groups = ops.w4_geometry(k, g)
    bound = (6 * padded // 64 + 2 * groups + 8) * 2.0 ** -23                 # as above
    assert ((got[rows].double() - exact).abs() <= bound * terms).all()


# The accumulators are kept in units of the current group's scale: scales that are zero, subnormal or tiny beside others, in
# the first, a middle and the last group, in all but one and in all of a column; signs that change; and large ones.
@pytest.mark.parametrize("k,g,zeros", [(1024, 64, "fractional"), (1152, 128, "integer"), (1536, 256, "fractional"), (1024, 128, "u4")])
def test_scales_far_apart(ops, k, g, zeros):
    m, n = 1409, 6144 if zeros == "u4" else 2820
    say(f"w4 forward, six-bit kernel, scales far apart: m={m} k={k} n={n} g={g} zero-points {zeros}")
    if zeros != "u4":
        assert ops.qmatmul_int4_block_takes(m, k, n, g)
    gen = torch.Generator(device="cuda").manual_seed(k + n)
    packed, scales, zp = ops.w4_quantize_pack(torch.randn(k, n, device="cuda", generator=gen) * 0.02, g)
    if zeros != "fractional":
        zp = zp.round().clamp(0, 15)
    col, last = 0, scales.shape[0] - 1
    for value in (1e-40, 1.4e-45, 1e-37, 1e-30, 0.0, -1e-39, -0.02, 1e25):
        for at in ([0], [last // 2], [last], [0, last], list(range(1, last)), list(range(last)), list(range(1, last + 1)), list(range(last + 1))):
            scales[at, col:col + 3] = value
            col += 5
    scales[::2, col:col + 40] *= 1e-33                   # back and forth
    scales[1::3, col + 20:col + 40] *= 1e-12
    scales[1, n - 7] = float("nan")
    x = torch.randn(m, k, device="cuda", generator=gen)
    x[m - 3] *= 1e8
    if zeros == "u4":
        shifts = 4 * torch.arange(8, device="cuda", dtype=torch.int32)
        qzeros = (zp.to(torch.int32).reshape(-1, n // 8, 8) << shifts).sum(2).to(torch.int32)
        got = ops.qmatmul_int4_zp4(x, packed, scales, qzeros, k, g)
    else:
        got = ops.qmatmul_int4(x, packed, scales, zp, k, g)
    rows = torch.cat([torch.arange(40), torch.arange(700, 740), torch.arange(m - 40, m)]).cuda()
    q = torch.stack([(packed >> (4 * i)) & 15 for i in range(8)], 1).reshape(-1, n)[:k].double()
    expand = lambda t: t.double().repeat_interleave(g, 0)[:k]
    z, s, xs = expand(zp), expand(scales), x[rows].double()
    exact = xs @ ((q - z) * s)
    near = z.round().clamp(0, 15)
    levels = xs.abs() @ ((q - near).abs() + (z - near).abs())
    terms = xs.abs() @ (((q - near).abs() + (z - near).abs()) * s.abs())
    # as above; a group far below the column's largest scale counts with 2^-60 of that, and with 2^-126 at least
    steps = -(-k // 64)
    bound = (6 * steps + 2 * scales.shape[0] + 8) * 2.0 ** -23 * terms + levels * (s.abs().amax(0) * 2.0 ** -59 + 2.0 ** -125)
    whole = torch.arange(n, device="cuda") != n - 7
    assert torch.equal(torch.isfinite(got), whole.expand(m, n))
    assert ((got[rows].double() - exact).abs() <= bound)[:, whole].all()


# Every st-th channel 2^p as large and met by weights of zero: the result is made of the small elements alone, whose bits must
# not suffer from their neighbours' size.  Error of the result as a whole.
@pytest.mark.parametrize("st", [2, 8, 32])
def test_small_elements_beside_large_channels(ops, st):
    m, k, n, g = 1500, 4096, 4096, 128
    assert ops.qmatmul_int4_block_takes(m, k, n, g)
    gen = torch.Generator(device="cuda").manual_seed(st)
    packed, scales, zp = ops.w4_quantize_pack(torch.randn(k, n, device="cuda", generator=gen) * 0.02, g)
    zp = zp.round().clamp(0, 15)
    expand = lambda t: t.double().repeat_interleave(g, 0)
    q = torch.stack([(packed >> (4 * i)) & 15 for i in range(8)], 1).reshape(k, n)
    q[::st] = expand(zp)[::st].to(torch.int32)
    shifts = (4 * torch.arange(8, device="cuda")).reshape(1, 8, 1)
    words = (q.reshape(k // 8, 8, n).long() << shifts).sum(1)
    packed = torch.where(words >= 2 ** 31, words - 2 ** 32, words).to(torch.int32)
    w = (q.double() - expand(zp)) * expand(scales)
    for p in (0, 3, 5, 6, 7, 8, 9, 10, 12, 16):
        say(f"w4 forward, six-bit kernel: every {st}. channel 2^{p} as large, weights of zero")
        x = torch.randn(m, k, device="cuda", generator=gen)
        x[:, ::st] *= 2.0 ** p
        exact = x.double() @ w
        err = ((ops.qmatmul_int4(x, packed, scales, zp, k, g).double() - exact).norm() / exact.norm()).item()
        say(f"    {err:.2e} of the result")
        # 22 bits of every element, and six additions per step of 64, each within 2^-24 of the result, independent of each other
        assert err <= 2.0 ** -22 + (6 * k / 64) ** 0.5 * 2.0 ** -24
