"""The projections of a prompt with RMSNorm, SwiGLU and the residual folded in (qmatmul_int4_block) against the same
operators one by one, at the edges of the kernels' tiles."""
import numpy as np
import pytest
import torch

import oracle
from gpu_util import dev, say
from rumus_amd import _lib, nn, ops

pytestmark = pytest.mark.gpu


# rows: blocks of 128 with a last one of 1, 60 or 128; columns: tiles of 256, 384 and 512 with and without an edge; k: an odd
# number of steps of 64, padded (1032 -> 1088, 1160 -> 1280) or not; 4, 2 and 1 per workgroup of the preparation
@pytest.mark.parametrize("m,k,n,g", [(1409, 1032, 2820, 64), (1408, 1024, 2816, 128), (1400, 1160, 6148, 128),
                                     (3516, 1088, 4100, 64), (1500, 4096, 4096, 128), (1500, 11008, 4096, 128)])
def test_folded_operators(m, k, n, g):
    assert ops.qmatmul_int4_block_takes(m, k, n, g)
    rng = np.random.default_rng(m + k + n)
    packed, scales, zp = ops.w4_quantize_pack(dev(rng.normal(0, 0.02, (k, n)).astype(np.float32)), g)
    res, bias = dev(rng.normal(0, 1, (m, n)).astype(np.float32)), dev(rng.normal(0, 1, n).astype(np.float32))
    x = rng.normal(0, 1, (m, 2 * k)).astype(np.float32)
    x[3:7, 33] *= 5000.0                       # runs that need further digits, in both halves
    x[m - 1, k + 100] *= 5000.0
    x[m - 2, 5] = np.nan
    x = dev(x)
    say(f"swiglu + residual m={m} k={k} n={n} g={g}")
    want = ops.add(ops.qmatmul_int4(ops.swiglu_rows(x), packed, scales, zp, k, g, bias=bias), res)
    got = ops.qmatmul_int4_block(x, packed, scales, zp, k, g, swiglu=True, bias=bias, residual=res)
    assert torch.equal(torch.nan_to_num(got, 1e30), torch.nan_to_num(want, 1e30)) and got[m - 2].isnan().all()
    aliased = res.clone()
    ops.qmatmul_int4_block(x, packed, scales, zp, k, g, swiglu=True, bias=bias, residual=aliased, out=aliased)
    assert torch.equal(torch.nan_to_num(aliased, 1e30), torch.nan_to_num(want, 1e30))

    say(f"rmsnorm m={m} k={k} n={n} g={g}")
    x1, w = x[:, :k].contiguous(), dev((1.0 + rng.normal(0, 0.1, k)).astype(np.float32))
    y = ops.rmsnorm(x1, w, 1e-5)
    want = ops.qmatmul_int4(y, packed, scales, zp, k, g)
    got = ops.qmatmul_int4_block(x1, packed, scales, zp, k, g, norm_weight=w, eps=1e-5)
    assert got[m - 2].isnan().all()
    keep = [r for r in range(m) if r != m - 2]
    # The sum of squares in another order moves a whole row by less than k / 64 roundings of 2^-24.  Every product with it is
    # rounded anew, and the matmul's sums of k / 64 steps with it (errors that grow like the root of their number): 64 in all
    a, b = got[keep].double(), want[keep].double()
    assert ((a - b).norm(dim=1) <= (k / 64 + 64) * 2.0 ** -24 * b.norm(dim=1)).all()
    say(f"residual alone m={m} k={k} n={n} g={g}")
    want = ops.add(ops.qmatmul_int4(y, packed, scales, zp, k, g), res)
    got = ops.qmatmul_int4_block(y, packed, scales, zp, k, g, residual=res)
    assert torch.equal(torch.nan_to_num(got, 1e30), torch.nan_to_num(want, 1e30))


def test_what_it_does_not_take_is_refused():
    packed, scales, zp = (dev(a) for a in oracle.w4_from_f32(np.ones((256, 64), np.float32), 64))
    assert not ops.qmatmul_int4_block_takes(4, 256, 64, 64) and not ops.qmatmul_int4_block_takes(4, 256, 64, 0)
    with pytest.raises(_lib.RumusError, match="block_takes"):
        ops.qmatmul_int4_block(torch.ones(4, 256, device="cuda"), packed, scales, zp, 256, 64)


# the four projections q|k|v, o, gate|up and down: the first and third large enough to fold; all of them; none
@pytest.mark.parametrize("heads,f,b,n,folded", [(8, 2816, 8, 500, [1, 0, 1, 0]), (16, 5504, 7, 512, [1, 1, 1, 0]), (8, 2816, 1, 100, [0] * 4)])
def test_prompt_block_equals_the_separate_operators(monkeypatch, heads, f, b, n, folded):
    say(f"decoder block, {heads} heads, prompt of {b} x {n} tokens, folded and not")
    gen = torch.Generator(device="cuda").manual_seed(2)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    d = heads * 128
    shapes = {"q": (d, d), "k": (d, d), "v": (d, d), "o": (d, d), "gate": (d, f), "up": (d, f), "down": (f, d)}
    block = nn.DecoderBlockW4.from_f32({name: rand(*s) * 0.02 for name, s in shapes.items()}, 128, heads)
    x = rand(b, n, d)
    taken = []
    folds = nn.DecoderBlockW4._folds_rows
    monkeypatch.setattr(nn.DecoderBlockW4, "_folds_rows", staticmethod(lambda *a: taken.append(folds(*a)) or taken[-1]))
    got = block(x)
    assert taken == [bool(t) for t in folded]
    monkeypatch.setattr(nn.DecoderBlockW4, "_folds_rows", staticmethod(lambda *a: False))
    for one, other in zip(got, block(x)):
        # two norms, each off by a few roundings of 2^-24, ahead of f32 sums
        assert one.shape == other.shape and (one - other).norm() <= 64 * 2.0 ** -24 * other.norm()


def test_captured_within_the_documented_workspace():
    m, k, n, g = 1500, 4096, 4096, 128
    say("qmatmul_int4_block captured in a graph, workspace of qmatmul_int4 reserved")
    gen = torch.Generator(device="cuda").manual_seed(3)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    packed, scales, zp = ops.w4_quantize_pack(rand(k, n) * 0.02, g)
    w, x, res = 1.0 + 0.1 * rand(k), rand(m, 2 * k), rand(m, n)
    x[3:7, 33] *= 5000.0
    x1 = x[:, :k].contiguous()
    calls = (lambda out: ops.qmatmul_int4_block(x, packed, scales, zp, k, g, swiglu=True, residual=res, out=out),
             lambda out: ops.qmatmul_int4_block(x1, packed, scales, zp, k, g, norm_weight=w, out=out))
    want = [call(None) for call in calls]
    side = torch.cuda.Stream()
    _lib.call("rumus_hip_workspace_reserve", side.cuda_stream, 5 * (m + 64) * (k + 128) + 1280)
    got = [torch.empty_like(t) for t in want]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        for call, out in zip(calls, got):
            call(out)
    for _ in range(3):
        for out in got:
            out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))
