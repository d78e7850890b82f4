"""Calls that are faster with more workspace than they need: what they take, and what they leave alone."""
import pytest

from gpu_util import free_workspaces, say

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def _weight(k, n, group, seed):
    import torch
    from rumus_amd import ops
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return ops.w4_quantize_pack(torch.empty((k, n), device="cuda").normal_(0.0, 0.02, generator=gen), group)


def _rows(m, k, seed):
    import torch
    return torch.empty((m, k), device="cuda").normal_(generator=torch.Generator(device="cuda").manual_seed(seed))


# digits of all rows at once (4.6 bytes per element) are more than the documented size for 385 x 3584, and more than the 32 MiB
# in which the f16 tiles run 1500 x 5120: such calls take their rows in two halves and have no room for codes
@pytest.mark.parametrize("m,k,n,reserve", [
    (385, 3584, 14336, 5 * (385 + 64) * (3584 + 128) + 1280), (1500, 5120, 4096, 32 * MIB)])
def test_reserved_size_is_kept(m, k, n, reserve):
    import torch
    from rumus_amd import _lib, ops
    say(f"qmatmul_int4 {m} x {k} -> {n} on a stream whose workspace is reserved")
    assert ops.qmatmul_int4_block_takes(m, k, n, 128)
    weight, x, y = _weight(k, n, 128, 1), _rows(m, k, 2), torch.empty((m, n), device="cuda")
    want = ops.qmatmul_int4(x, *weight, k, 128)
    # and with a block's operators around it, which have to find the second half's rows of the gate, the values and the residual
    gate, res, z = _rows(m, 2 * k, 3), _rows(m, n, 4), torch.empty_like(y)
    folded = lambda out: ops.qmatmul_int4_block(gate, *weight, k, 128, swiglu=True, residual=res, out=out)
    want_folded = folded(None)
    free_workspaces()
    stream = torch.cuda.Stream()
    _lib.call("rumus_hip_workspace_reserve", stream.cuda_stream, reserve)
    with torch.cuda.stream(stream):
        ops.qmatmul_int4(x, *weight, k, 128, out=y)
        folded(z)
    stream.synchronize()
    assert torch.equal(y, want) and torch.equal(z, want_folded)
    assert free_workspaces() <= reserve + 4 * MIB                 # (memory comes in 2 MiB, give or take as much); the codes are 15 MB and more


def test_a_graph_keeps_its_workspace():
    """A call that lets the workspace grow for speed leaves the memory of a graph that was captured on the stream before."""
    import torch
    from rumus_amd import ops
    k = 4096
    say("qmatmul_int4 1500 x 4096 -> 4096 in a graph, 1200 x 4096 -> 11008 beside it on the graph's stream")
    small, large = _weight(k, 4096, 128, 1), _weight(k, 11008, 128, 2)
    x, other = _rows(1500, k, 3), _rows(1200, k, 4)
    want, beside = ops.qmatmul_int4(x, *small, k, 128), ops.qmatmul_int4(other, *large, k, 128)
    free_workspaces()
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    y, got = torch.empty_like(want), torch.empty_like(beside)
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        ops.qmatmul_int4(x, *small, k, 128, out=y)
    stream.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        ops.qmatmul_int4(x, *small, k, 128, out=y)
    with torch.cuda.stream(stream):
        ops.qmatmul_int4(other, *large, k, 128, out=got)
    stream.synchronize()
    assert torch.equal(got, beside)
    for _ in range(2):
        y.zero_()
        graph.replay()
        with torch.cuda.stream(stream):
            got.zero_()
            ops.qmatmul_int4(other, *large, k, 128, out=got)
        torch.cuda.synchronize()
        assert torch.equal(y, want) and torch.equal(got, beside)
    # 1500 rows: digits and sums, 29 MB, and the codes of 4096 columns, 13 MB; beside that 23 MB and 34 MB for the other call
    assert free_workspaces() >= 92 * MIB


def test_growing_for_speed_is_bounded():
    """Streams do not keep more than 256 MiB of earlier workspaces: then a call does without."""
    import torch
    from rumus_amd import ops
    m, k = 8192, 4096
    say("qmatmul_int4 8192 x 4096 -> 4096 and on to 14336 columns on one stream")
    x = _rows(m, k, 3)
    stream = torch.cuda.Stream()
    weights = [_weight(k, n, 128, n) for n in (4096, 8192, 11008, 14336)]
    want = [ops.qmatmul_int4(x, *w, k, 128) for w in weights]
    free_workspaces()
    for w, y in zip(weights, want):
        with torch.cuda.stream(stream):
            got = ops.qmatmul_int4(x, *w, k, 128)
        stream.synchronize()
        assert torch.equal(got, y)
    # digits and sums take 147 MiB, the codes 12, 24, 32 and 42: the first growth keeps 160 MiB beside 172, a second would keep 332
    assert 320 * MIB <= free_workspaces() <= 356 * MIB


def test_growing_beside_a_capture():
    """While another stream is being captured a call may still let its workspace grow for speed."""
    import torch
    from rumus_amd import _lib, ops
    k = 4096
    say("qmatmul_int4 1200 x 4096 -> 11008 while another stream is captured")
    small, large = _weight(k, 4096, 128, 1), _weight(k, 11008, 128, 2)
    x, other = _rows(1500, k, 3), _rows(1200, k, 4)
    beside = ops.qmatmul_int4(other, *large, k, 128)
    free_workspaces()
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    got, doubled = torch.empty_like(beside), torch.empty_like(x)
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        ops.qmatmul_int4(x, *small, k, 128, out=torch.empty((1500, 4096), device="cuda"))
    stream.synchronize()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        torch.mul(x, 2.0, out=doubled)
        with torch.cuda.stream(stream):
            ops.qmatmul_int4(other, *large, k, 128, out=got)
    stream.synchronize()
    assert torch.equal(got, beside)
    for _ in range(2):
        doubled.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(doubled, 2.0 * x)
    assert free_workspaces() >= 50 * MIB                          # digits of 1200 rows, 24 MB, and the codes, 34 MB


def _captured_in(reserve, call, outs):
    """The outputs of a call captured on a stream with a workspace of `reserve` bytes, after each of three replays."""
    import torch
    from rumus_amd import _lib
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    _lib.call("rumus_hip_workspace_reserve", stream.cuda_stream, reserve)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        call()
    for _ in range(3):
        outs.zero_()
        graph.replay()
        torch.cuda.synchronize()
        yield outs


def test_q8_with_a_ragged_k_needs_no_partial_sums():
    """One block per column: the int8 GEMM inside has no room for shares of K, in a capture on a workspace of what the call keeps there."""
    import torch
    from rumus_amd import ops
    m, k, n = 384, 2064, 500
    say(f"matmul_q8 {m} x {k} x {n}, one block per column, captured without room for shares of K")
    a, w = _rows(m, k, 3), _rows(n, k, 4)
    words = ops.q8_quantize(w.reshape(-1), k)
    wq, sw = ops.q8_dense_layout(words, k, n, k)
    up = lambda v: -(-v // 256) * 256
    own = up(4 * m * k) + up(16 * m) + up(16 * m * n)            # digit planes, their factors, the planes' products
    c = torch.empty((m, n), device="cuda")
    for room, call in ((own + up(n * k) + up(4 * n), lambda out: ops.matmul_q8(a, words, k, n, k, out=out)),
                       (own, lambda out: ops.matmul_q8_dense(a, wq, sw, out=out))):
        want = call(torch.empty_like(c))
        for got in _captured_in(room, lambda: call(c), c):
            assert torch.equal(got, want)


# 100 rows: eight shares of n fit, sixteen would be faster; 40 rows with a short n: four fit
@pytest.mark.parametrize("m,k,n,shares", [(100, 512, 11008, 8), (40, 512, 2048, 4), (100, 2048, 1028, 2), (32, 4096, 1028, 2)])
def test_grad_x_with_room_for_fewer_shares(m, k, n, shares):
    import torch
    from rumus_amd import ops
    say(f"qmatmul_int4_t {m} rows of {n} -> {k}, captured with room for {shares} shares of n")
    packed, scales, zp = _weight(k, n, 128, 5)
    gy = _rows(m, n, 6)
    out = torch.empty((m, k), device="cuda")
    up = lambda v: -(-v // 256) * 256
    entries = k // 128 * n
    room = up(4 * m) + up(4 * (k // 128)) + 2 * up(4 * entries) + up(2 * entries + 64) + shares * m * k * 4
    q = torch.stack([(packed.view(torch.int32) >> (4 * i)) & 15 for i in range(8)], 1).reshape(k, n).double()
    each = lambda t: t.double().repeat_interleave(128, 0)
    w = ((q - each(zp)) * each(scales)).t().contiguous()
    want, size = gy.double() @ w, gy.double().abs() @ w.abs()
    for got in _captured_in(room, lambda: ops.qmatmul_int4_t(gy, packed, scales, zp, k, 128, out=out), out):
        # test_gpu_w4_t_wide.py's bound of an ordinary sum, far above both share counts' rounding
        assert float(((got.double() - want).abs() / size).max()) < 2e-6


# the plan of 256 columns a workgroup wants more shares of K than that of 512, for which there is room; stages of 128 k of each of these
@pytest.mark.parametrize("m,k,n,shares,stages", [(257, 4096, 768, 11, 3), (540, 2048, 768, 6, 3)])
def test_f16_tiles_with_room_for_fewer_shares(m, k, n, shares, stages):
    import torch
    from rumus_amd import ops
    say(f"qmatmul_int4 {m} x {k} -> {n}, groups of 32, captured with room for {shares} shares of K")
    packed, scales, zp = _weight(k, n, 32, 5)
    x, out = _rows(m, k, 6), torch.empty((m, n), device="cuda")
    room = 1024 + -(-8 * m // 256) * 256 + shares * m * n * 4      # flags, the rows' factors, partial tiles
    q = torch.stack([(packed.view(torch.int32) >> (4 * i)) & 15 for i in range(8)], 1).reshape(k, n).double()
    each = lambda t: t.double().repeat_interleave(32, 0)
    w = (q - each(zp)) * each(scales)
    want, size = x.double() @ w, x.double().abs() @ w.abs()
    for got in _captured_in(room, lambda: ops.qmatmul_int4(x, packed, scales, zp, k, 32, out=out), out):
        # f32 additions: eight steps a stage, two products each, a settlement every two, then the shares; zero-points up to half a step off
        assert float(((got.double() - want).abs() / size).max()) < (20 * stages + shares + 16) * 2.0 ** -24


# few rows on which the integer kernel is the faster one, and needs workspace: eight of two rounds of workgroups, wide row-major arrays, act-order
@pytest.mark.parametrize("m,k,n,group,form", [(6, 3200, 9600, 64, "plain"), (8, 7168, 4416, 128, "plain"), (3, 4096, 12288, 64, "plain"),
                                              (4, 4096, 12288, 64, "half"), (8, 2048, 8192, 128, "act"), (5, 2560, 8704, 32, "plain")])
def test_few_rows_without_workspace(m, k, n, group, form):
    import torch
    from rumus_amd import ops
    say(f"qmatmul_int4 {m} x {k} -> {n}, groups of {group}, {form}, captured without workspace")
    packed, scales, zp = _weight(k, n, group, 5)
    x = _rows(m, k, 6).to(torch.float16 if form == "half" else torch.float32)
    out = torch.empty((m, n), dtype=x.dtype, device="cuda")
    perm = torch.randperm(k, generator=torch.Generator(device="cuda").manual_seed(7), device="cuda").to(torch.int32)
    call = {"plain": lambda: ops.qmatmul_int4(x, packed, scales, zp, k, group, out=out),
            "half": lambda: ops.qmatmul_int4_f16(x, packed, scales, zp, k, group, out=out),
            "act": lambda: ops.qmatmul_int4_perm(x, packed, scales, zp, k, group, perm=perm, out=out)}[form]
    q = torch.stack([(packed.view(torch.int32) >> (4 * i)) & 15 for i in range(8)], 1).reshape(k, n).double()
    each = lambda t: t.double().repeat_interleave(group, 0)
    w, rows = (q - each(zp)) * each(scales), (x[:, perm.long()] if form == "act" else x).double()
    want, size = rows @ w, rows.abs() @ w.abs() + rows.abs().amax(1, keepdim=True) * w.abs().sum(0)
    free_workspaces()
    for got in _captured_in(0, call, out):
        # test_gpu_w4_few_rows.py's bound; one rounding to f16
        assert float(((got.double() - want).abs() / size).max()) < (2.0 ** -11 if form == "half" else 2.0 ** -20)
