"""INT8 GEMM with K that ends in one to three chunks of 16: every tile size, exact i32 sums."""
import pytest

from gpu_util import free_workspaces, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n", [
    (9, 1424, 100), (32, 1568, 1000), (100, 1840, 64), (60, 4144, 520),    # one-wave tiles, whole K and K in shares
    (64, 1728, 11008), (64, 1744, 11008), (64, 1728, 10752),               # to either side of the line for large outputs
    (130, 2064, 300), (300, 4128, 260), (257, 2096, 1000),                 # 128 x 128 tiles, the same
    (4096, 2064, 4100), (4090, 2080, 4224), (4096, 2096, 4128),            # 256 x 128 tiles
    (33, 1008, 70), (9, 1040, 100), (100, 1072, 64), (300, 1552, 200), (300, 80, 200), (2048, 208, 2304)])                    # shorter: register-staged tiles
def test_tail_of_k(m, k, n):
    import torch
    from rumus_amd import ops
    say(f"i8_gemm m={m} k={k} n={n}")
    gen = torch.Generator(device="cuda").manual_seed(m + k + n)
    x, w = (torch.randint(-128, 128, (r, k), generator=gen, device="cuda", dtype=torch.int32) for r in (m, n))
    sx, sw, bias = (torch.rand(r, generator=gen, device="cuda") + 0.5 for r in (m, n, n))
    y, acc = ops.i8_gemm(x.to(torch.int8), w.to(torch.int8), sx, sw, bias, want_acc=True)
    want = x.double() @ w.double().t().contiguous()                        # below 2^53: exact
    assert torch.equal(acc.double(), want)
    assert torch.equal(y, want.float() * sx[:, None] * sw + bias)    # each operation rounded by itself
    y, _ = ops.i8_gemm(x.to(torch.int8), w.to(torch.int8), sx, sw, bias)
    assert torch.equal(y, want.float() * sx[:, None] * sw + bias)


def test_tail_without_room_for_shares():
    """A stream whose workspace the caller sized, too small for partial sums, and a capture on one without any: the same sums."""
    import torch
    from rumus_amd import _lib, ops
    say("i8_gemm 60 x 4144 x 520 with no room for partial sums")
    gen = torch.Generator(device="cuda").manual_seed(3)
    x, w = (torch.randint(-128, 128, (r, 4144), generator=gen, device="cuda", dtype=torch.int32).to(torch.int8) for r in (60, 520))
    _, want = ops.i8_gemm(x, w, want_acc=True, want_y=False)
    big, wide = torch.cat([x] * 2), torch.cat([w] * 4)
    assert _lib.lib().rumus_hip_i8_gemm_workspace_size(120, 4144, 2080) >= 3 << 20
    free_workspaces()
    sized, captured = torch.cuda.Stream(), torch.cuda.Stream()
    _lib.call("rumus_hip_workspace_reserve", sized.cuda_stream, 256)   # a mebibyte
    with torch.cuda.stream(sized):
        _, got = ops.i8_gemm(big, wide, want_acc=True, want_y=False)
    sized.synchronize()
    assert torch.equal(got, torch.cat([torch.cat([want] * 4, 1)] * 2))
    assert free_workspaces() <= 4 << 20                          # (memory comes in 2 MiB, give or take as much)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=captured):
        _, got = ops.i8_gemm(x, w, want_acc=True, want_y=False)
    for _ in range(3):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
