"""Large batches of the INT4 forward with the weights converted once per call, and by every block of rows for itself (a workspace
of the caller's own size, with no room for the codes): the same bits, and the product in float64."""
import pytest

from gpu_util import free_workspaces, say

pytestmark = pytest.mark.gpu

MIB = 1 << 20


# every width of the workgroups' columns, groups of one, two and three steps of 64 k, an odd number of steps, K no multiple of the
# group, a last block of rows and columns with little in it, both forms of the zero-points, columns across two words of packed ones
@pytest.mark.parametrize("m,k,n,group,packed_zero", [
    (1024, 2112, 6148, 64, False), (1400, 3072, 4104, 64, True), (600, 4096, 11016, 128, False), (1500, 3000, 3300, 192, False), (1536, 2112, 5512, 64, True), (1300, 4096, 11016, 128, True),
    (2049, 4096, 4100, 128, False), (3000, 1024, 2824, 128, True), (2048, 2056, 5504, 256, False), (4096, 1088, 2820, 64, False)])
def test_codes_once_or_by_every_block(m, k, n, group, packed_zero):
    import torch
    from rumus_amd import _lib, ops
    assert ops.qmatmul_int4_block_takes(m, k, n, group)
    say(f"qmatmul_int4 m={m} k={k} n={n} g={group} packed zero-points {packed_zero}, with and without room for the codes")
    gen = torch.Generator(device="cuda").manual_seed(m + n)
    w = torch.empty((k, n), device="cuda").normal_(0.0, 0.02, generator=gen)
    packed, scales, zp = ops.w4_quantize_pack_awq(w, group) if packed_zero else ops.w4_quantize_pack(w, group)
    x = torch.empty((m, k), device="cuda").normal_(generator=gen)
    x[::7, ::37] *= 3000.0                                       # marked runs in some rows
    call = ops.qmatmul_int4_zp4 if packed_zero else ops.qmatmul_int4
    padded, groups = ops.w4_geometry(k, group)
    blocks, steps = -(-m // 128), padded // 64                   # digits, exponents, sums, row factors, column scales, flags
    digits = blocks * (steps * (36864 + 512) + -(-steps // 2) * 512 + 1024) + 4 * n + 1024 + 512
    codes = 48 * n * steps                                       # and more where the last block of columns is not full
    outs = []
    for sized in (False, True):
        free_workspaces()
        stream = torch.cuda.Stream()
        if sized:
            _lib.call("rumus_hip_workspace_reserve", stream.cuda_stream, digits)
        with torch.cuda.stream(stream):
            outs.append(call(x, packed, scales, zp, k, group))
        stream.synchronize()
        took = free_workspaces()
        # memory comes in 2 MiB, and what others of that size hold blurs it by as much: the smallest codes do not show
        if codes > 6 * MIB:
            assert took <= digits + 4 * MIB if sized else took >= digits + codes - 3 * MIB
    assert torch.equal(outs[0].view(torch.int32), outs[1].view(torch.int32))
    q = torch.stack([(packed.view(torch.int32) >> (4 * i)) & 15 for i in range(8)], 1).reshape(padded, n).double()
    if packed_zero:
        zp = torch.stack([(zp.view(torch.int32) >> (4 * i)) & 15 for i in range(8)], 2).reshape(groups, n)
    each = lambda t: t.double().repeat_interleave(group, 0)
    want = x.double() @ ((q - each(zp)) * each(scales))[:k]
    # f32 sums of k terms, rounded in blocks of 64 k: far below k half ulps of the summed magnitudes
    size = x.double().abs() @ ((q - each(zp)).abs() * each(scales).abs())[:k]
    assert float(((outs[0].double() - want).abs() / size).max()) < 2e-6
