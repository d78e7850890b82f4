"""The native front end of the frequent calls (csrc/host_calls.cpp) against the general path in ops.py: same results where it
takes the call, the general path's answer or error where it does not."""
import pytest
import torch

from gpu_util import say
from rumus_amd import _lib, nn, ops

K, N, G = 256, 64, 64


def _operands(rows=3):
    gen = torch.Generator(device="cuda").manual_seed(5)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    packed, scales, zp = ops.w4_quantize_pack(rand(K, N), G)
    w8 = nn.Int8Linear.from_linear(nn.Linear(rand(K, N)))
    q8 = nn.quantize(rand(K, N), 32)
    perm = torch.randperm(K, device="cuda", generator=gen).to(torch.int32)
    d = {"x": rand(rows, K), "gy": rand(rows, N), "bias": rand(N), "w4": (packed, scales, zp), "perm": perm,
         "decode": ops.w4_decode_layout(packed, scales, zp, G), "w8": w8, "q8": q8, "norm": rand(K), "res": rand(rows, N),
         "gu": rand(rows, 2 * K)}
    qkv = rand(2, 1, 3, 4, 128)
    d["att"] = (qkv[:, :, 0], qkv[:, :, 1], qkv[:, :, 2], rand(2, 40, 4, 128), rand(2, 40, 4, 128))
    return d


def _calls(d):
    x, w4, dec = d["x"], d["w4"], d["decode"]
    out = torch.empty((x.shape[0], N), device="cuda")
    return {
        "int4": lambda: ops.qmatmul_int4(x, *w4, K, G, bias=d["bias"]),
        "int4 out": lambda: ops.qmatmul_int4(x, *w4, K, G, out=out),
        "int4 f16": lambda: ops.qmatmul_int4_f16(x.half(), *w4, K, G, bias=d["bias"]),
        "int4 perm": lambda: ops.qmatmul_int4_perm(x, *w4, K, G, perm=d["perm"]),
        "int4 static": lambda: ops.qmatmul_int4_perm_static(x, *w4, K, G, perm=d["perm"], out=out),
        "int4 decode": lambda: ops.qmatmul_int4_decode(x, *dec, K, G, bias=d["bias"]),
        "int4 t": lambda: ops.qmatmul_int4_t(d["gy"], *w4, K, G),
        "int4 block": lambda: ops.qmatmul_int4_decode_block(x, *dec, K, G, norm_weight=d["norm"], residual=d["res"]),
        "int4 block swiglu": lambda: ops.qmatmul_int4_decode_block(d["gu"], *dec, K, G, swiglu=True, bias=d["bias"]),
        "q8": lambda: ops.matmul_q8(x, d["q8"].buffer, K, N, 32),
        "q8 f16": lambda: ops.matmul_q8_f16(x.half(), d["q8"].buffer, K, N, 32),
        "int8": lambda: ops.i8_linear(x, d["w8"].wq, d["w8"].sw, d["bias"]),
        "int8 no contiguous rows": lambda: ops.i8_linear(d["gu"][:, :K], d["w8"].wq, d["w8"].sw),
        "attention": lambda: ops.attention_decode_append(*d["att"], 17),
        "no rows": lambda: ops.qmatmul_int4(x[:0], *w4, K, G),
    }


@pytest.mark.gpu
def test_native_calls_equal_the_general_path(monkeypatch):
    d = _operands()
    stream = torch.cuda.Stream()
    native = ops._native
    taken = []

    def watch(name, *args):
        y = native(name, *args)
        taken.append(y is not None)
        return y

    for name, call in _calls(d).items():
        say(f"native call: {name}")
        monkeypatch.setattr(ops, "_native", watch)
        taken.clear()
        got = call().clone()
        assert taken == [name not in ("int8 no contiguous rows", "no rows")], name
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            side = call().clone()
        stream.synchronize()
        monkeypatch.setattr(ops, "_native", lambda *a: None)
        want = call()
        assert got.dtype == want.dtype and torch.equal(got, want) and torch.equal(side, want), name


@pytest.mark.gpu
def test_refusals_are_those_of_the_general_path(monkeypatch):
    d = _operands()
    x, (p, s, z) = d["x"], d["w4"]
    cases = [
        (TypeError, lambda: ops.qmatmul_int4(x.double(), p, s, z, K, G)),
        (TypeError, lambda: ops.qmatmul_int4(x.cpu(), p, s, z, K, G)),
        (ValueError, lambda: ops.qmatmul_int4(x.t().contiguous().t(), p, s, z, K, G)),
        (ValueError, lambda: ops.qmatmul_int4(x[:, :8].contiguous(), p, s, z, K, G)),
        (ValueError, lambda: ops.qmatmul_int4(x, p, s[:1], z, K, G)),
        (ValueError, lambda: ops.qmatmul_int4(x, p, s, z, K, G, bias=d["bias"][:8])),
        (ValueError, lambda: ops.qmatmul_int4_perm(x, p, s, z, K, G, perm=d["perm"][:8])),
        (ValueError, lambda: ops.qmatmul_int4(x, p, s, z, K, G, out=torch.empty((4, N), device="cuda"))),
        (_lib.RumusError, lambda: ops.qmatmul_int4(x[:, :240].contiguous(), p, s, z, 240, 60)),
        (ValueError, lambda: ops.qmatmul_int4_t(x, p, s, z, K, G)),
        (ValueError, lambda: ops.matmul_q8(x, d["q8"].buffer[:9], K, N, 32)),
        (ValueError, lambda: ops.i8_linear(x, d["w8"].wq, d["w8"].sw[:3])),
        (ValueError, lambda: ops.i8_linear(x[:, :16].contiguous(), d["w8"].wq, d["w8"].sw)),
        (_lib.RumusError, lambda: ops.attention_decode_append(*d["att"], 40)),
    ]
    for i, (kind, call) in enumerate(cases):
        say(f"refused call {i}")
        with pytest.raises(kind) as got:
            call()
        with monkeypatch.context() as m:
            m.setattr(ops, "_native", lambda *a: None)
            with pytest.raises(kind) as want:
                call()
        assert str(got.value) == str(want.value)


def test_what_is_not_plain_is_left_to_the_general_path():
    host = _lib.host()
    t = torch.zeros(2, 256)
    assert host.rumus_hip_qmatmul_int4(t, t, t, t, None, None, 256, 64, None) is None
    assert host.rumus_hip_qmatmul_int4() is None
    assert host.int8_linear(t, t, t, None) is None
    assert host.matmul_q8(t, t, 256, 2, 2 ** 70) is None
    assert host.attention_decode_append(t, t, t, t, t, -1) is None
