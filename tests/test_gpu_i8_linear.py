"""The W8A8 layer in one call against its two halves: one launch for few rows, the same bits everywhere."""
import pytest
import torch

from gpu_util import say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from rumus_amd import ops
    return ops


def operands(m, k, n, seed=0):
    gen = torch.Generator().manual_seed(m * 7919 + k * 31 + n + seed)
    x = torch.randn((m, k), generator=gen)
    x[:, 0] *= 20.0
    wq = torch.randint(-128, 128, (n, k), generator=gen, dtype=torch.int8)
    return x.cuda(), wq.cuda(), torch.rand(n, generator=gen).cuda(), torch.randn(n, generator=gen).cuda()


# the rows that share a wave or take several, each K's number of loads a lane, ragged last steps, fewer steps than waves, one tile and
# several a workgroup (n > 4096), a last tile of one column, and the sizes just past what one launch takes
@pytest.mark.parametrize("m,k,n", [
    (1, 16, 1), (1, 64, 16), (1, 4096, 33), (1, 4112, 70), (1, 8208, 48), (1, 16384, 20), (1, 16400, 20), (1, 1008, 9000),
    (2, 48, 17), (2, 4096, 4113), (2, 8192, 32), (2, 16384, 16), (2, 11008, 4112),
    (3, 2048, 100), (3, 2064, 40), (4, 4112, 24), (4, 8192, 8208), (4, 8208, 24),
    (5, 1024, 65), (6, 1040, 31), (8, 4096, 4100), (8, 4080, 12), (7, 4112, 12), (8, 528, 12000),
    (2, 3088, 8200), (2, 3072, 8200), (9, 1024, 50), (13, 512, 2048), (16, 2048, 5000), (16, 1040, 18), (16, 2064, 18), (12, 16, 5), (17, 512, 64)])
def test_i8_linear_equals_its_halves(ops, m, k, n):
    say(f"i8_linear m={m} k={k} n={n}")
    x, wq, sw, bias = operands(m, k, n)
    if m > 1:
        x[1] = 0.0
    for b in (None, bias):
        xq, sx = ops.i8_quantize_rows(x)
        want, _ = ops.i8_gemm(xq, wq, sx, sw, b)
        assert torch.equal(ops.i8_linear(x, wq, sw, b), want)


def test_i8_linear_rows_that_are_not_finite(ops):
    say("i8_linear with NaN and infinities")
    x, wq, sw, _ = operands(6, 1040, 40)
    x[0, 3], x[2, 1039], x[4, 5], x[5] = float("nan"), float("inf"), 1e-42, -0.0
    xq, sx = ops.i8_quantize_rows(x)
    want, _ = ops.i8_gemm(xq, wq, sx, sw)
    assert torch.equal(torch.nan_to_num(ops.i8_linear(x, wq, sw), nan=7.0), torch.nan_to_num(want, nan=7.0))


# 127 / 1e-37 is an infinity: what stands between the end of a row and that of its last step of 64 has to be zero all the same
@pytest.mark.parametrize("m,k,n", [(1, 80, 40), (1, 8208, 20), (2, 1040, 33), (3, 4112, 17), (5, 1040, 40), (8, 2064, 33), (12, 16, 5), (16, 1040, 18)])
def test_i8_linear_rows_of_tiny_values(ops, m, k, n):
    say(f"i8_linear m={m} k={k} n={n}, rows of 1e-37")
    x, wq, sw, bias = operands(m, k, n)
    x[::2] = 1e-37
    xq, sx = ops.i8_quantize_rows(x)
    for b in (None, bias):
        want, _ = ops.i8_gemm(xq, wq, sx, sw, b)
        assert torch.equal(ops.i8_linear(x, wq, sw, b), want)


def test_i8_linear_from_rows_of_any_alignment(ops):
    say("i8_linear, x at an odd float")
    x, wq, sw, bias = operands(3, 528, 200)
    odd = torch.empty(3 * 528 + 1, device="cuda")[1:].view(3, 528)
    odd.copy_(x)
    assert torch.equal(ops.i8_linear(odd, wq, sw, bias), ops.i8_linear(x, wq, sw, bias))


def test_i8_linear_replays_in_a_graph(ops):
    say("i8_linear captured")
    x, wq, sw, bias = operands(8, 2064, 300)
    ops.i8_linear(x, wq, sw, bias)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = ops.i8_linear(x, wq, sw, bias)
    for seed in range(3):
        x.copy_(operands(8, 2064, 300, seed + 1)[0])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, ops.i8_linear(x, wq, sw, bias))
