"""The int8 matrix-core kernel at every size of its workgroups' tiles (rows, columns per lane), against float64."""
import pytest

from gpu_util import say

pytestmark = pytest.mark.gpu


def _check(m, k, n, group, packed_zero, x):
    import torch
    from rumus_amd import ops
    gen = torch.Generator(device="cuda").manual_seed(m + n)
    w = torch.empty((k, n), device="cuda").normal_(0.0, 0.02, generator=gen)
    packed, scales, zp = ops.w4_quantize_pack_awq(w, group) if packed_zero else ops.w4_quantize_pack(w, group)
    y = (ops.qmatmul_int4_zp4 if packed_zero else ops.qmatmul_int4)(x, packed, scales, zp, k, group)
    padded, groups = ops.w4_geometry(k, group)
    q = torch.stack([(packed.view(torch.int32) >> (4 * i)) & 15 for i in range(8)], 1).reshape(padded, n).double()
    if packed_zero:
        zp = torch.stack([(zp.view(torch.int32) >> (4 * i)) & 15 for i in range(8)], 2).reshape(groups, n)
    each = lambda t: t.double().repeat_interleave(group, 0)
    exact, z, s = x.double(), each(zp)[:k], each(scales)[:k]
    want = exact @ ((q[:k] - z) * s)
    # x in fixed point, within 2^-22 of a row's largest magnitude, against the whole nibble and the zero-point; and the f32 sums:
    # a rounding of 2^-24 per chunk of 64 or 128 k and per share of K, of the summed magnitudes
    fixed = exact.abs().amax(1, keepdim=True) * ((q[:k] + z.abs()) * s.abs()).sum(0) * 2.0 ** -22
    sums = exact.abs() @ ((q[:k] + z.abs()) * s.abs()) * (2 * (padded // 64) + 8) * 2.0 ** -24
    assert bool(((y.double() - want).abs() <= fixed + sums).all())
    assert float((y.double() - want).norm() / want.norm()) < 2e-6


# rows and columns of a workgroup: 16 to 64 and 16 to 64; last blocks with little in them, K no multiple of the group
@pytest.mark.parametrize("m,k,n", [
    (9, 1000, 20), (15, 2048, 5004), (9, 256, 11016), (10, 1000, 16392), (17, 1000, 4096), (31, 2048, 8200), (17, 256, 11016),
    (65, 1000, 5000), (47, 256, 4104), (33, 1000, 8200), (47, 2048, 11016), (33, 256, 16392), (100, 1000, 4104), (113, 2048, 5000),
    (100, 256, 8200), (128, 6144, 4096)])
@pytest.mark.parametrize("group,packed_zero", [(64, False), (128, False), (128, True)])
def test_tiles(m, k, n, group, packed_zero):
    import torch
    if packed_zero:
        n = n // 8 * 8
    say(f"qmatmul_int4 m={m} k={k} n={n} g={group} packed zero-points {packed_zero}")
    gen = torch.Generator(device="cuda").manual_seed(m * k)
    _check(m, k, n, group, packed_zero, torch.empty((m, k), device="cuda").normal_(generator=gen))


# the last share of K holds 16 elements (912), 8 (4104) and 40 (1000)
@pytest.mark.parametrize("m,k,n", [(32, 912, 5504), (20, 4104, 516), (48, 1000, 1028)])
def test_short_last_share(m, k, n):
    import torch
    say(f"qmatmul_int4 m={m} k={k} n={n}: a share of few elements, with and without towers in it")
    gen = torch.Generator(device="cuda").manual_seed(m * k)
    x = torch.empty((m, k), device="cuda").normal_(generator=gen)
    _check(m, k, n, 64, False, x)
    x[::3, k - 2] = 3000.0                                       # one element of the last share above the rest
    _check(m, k, n, 64, False, x)


# shares of 1 to 31 elements at the end of K (897 .. 927; groups of 128: 1032), most of their elements 2^20 (f16: 2^12) above the rest and met
# by weights of zero: what the small ones say stays, as it would with every large element multiplied by itself in f32
@pytest.mark.parametrize("k,group", [(897, 64), (904, 64), (909, 64), (912, 64), (920, 64), (927, 64), (1032, 128)])
@pytest.mark.parametrize("half", [False, True])
def test_short_share_of_two_heights(k, group, half):
    import torch
    from rumus_amd import ops
    m, n, begin = 37, 1032, k // 64 * 64
    towers = slice(begin, begin + min((k - begin) * 5 // 8, 16))
    say(f"qmatmul_int4 m={m} k={k} n={n} g={group} f16 {half}: a share of {k - begin} elements, {towers.stop - begin} of them towers")
    gen = torch.Generator(device="cuda").manual_seed(k)
    w = torch.empty((k, n), device="cuda").normal_(0.0, 0.02, generator=gen)
    x = torch.zeros((m, k), device="cuda")
    x[:, begin:].normal_(generator=gen)
    x[:, towers] *= 2.0 ** 12 if half else 2.0 ** 20
    w[towers] = 0.0
    if half:
        x = x.half().float()
    x[5, k - 1], x[33, begin] = float("inf"), float("nan")
    packed, scales, zp = ops.w4_quantize_pack(w, group, symmetric=True)      # (a weight of zero is the zero-point itself)
    y = ops.qmatmul_int4_f16(x.half(), packed, scales, zp, k, group) if half else ops.qmatmul_int4(x, packed, scales, zp, k, group)
    padded, groups = ops.w4_geometry(k, group)
    q = torch.stack([(packed.view(torch.int32) >> (4 * i)) & 15 for i in range(8)], 1).reshape(padded, n).double()
    assert not y[[5, 33]].isfinite().any()                       # and no other row is touched by them
    x[[5, 33]], y[[5, 33]] = 0.0, 0.0
    small, s = x.double(), scales.double().repeat_interleave(group, 0)[:k]
    small[:, towers] = 0.0
    want = small @ ((q[:k] - 8.0) * s)
    # the small ones: exact, or in fixed point within 2^-22 of their largest, against the whole nibble and the zero-point; sums of
    # their products, each of two roundings, in f32; f16 results one rounding more
    bound = small.abs().amax(1, keepdim=True) * ((q[begin:k] + 8.0) * s[begin:].abs()).sum(0) * 2.0 ** -22
    bound += small.abs() @ ((q[:k] - 8.0).abs() * s.abs()) * 40 * 2.0 ** -24
    if half:
        bound += want.abs() * 2.0 ** -11 + 2.0 ** -25
    assert bool(((y.double() - want).abs() <= bound).all())
