"""The work a user of the quantized layers has this library do, as cases to time.

A case is one pass through the public modules (``rumus_amd.nn``): an INT4 layer (``kind`` "linear", with its input
gradient when ``backward``), a W8A8 layer ("int8"), the block-format INT8 matmul ("q8"), the quantizers that make
those weights ("quantize") and a decoder block built from INT4 projections ("block", one token against a cache when
``pos`` > 0, a prompt otherwise).  ``listed`` names the fixed ones, ``draw`` gives more over the same ranges,
``prepare`` makes what the program holds before the call, ``run`` is the call, ``work`` what it cannot do without.
"""
from __future__ import annotations

import math

import torch

from rumus_amd import nn, ops


# ---- the cases -----------------------------------------------------------------------------

def _linear(rows, k, n, group=128, *, order="plain", zero="float", act="f32", bias=False, backward=False):
    return {"kind": "linear", "rows": rows, "k": k, "n": n, "group": group, "order": order, "zero": zero, "act": act,
            "bias": bias, "backward": backward}


def _int8(rows, k, n, bias=False):
    return {"kind": "int8", "rows": rows, "k": k, "n": n, "bias": bias}


def _q8(rows, k, n, block, act="f32", dense=False):
    return {"kind": "q8", "rows": rows, "k": k, "n": n, "block": block, "act": act, "dense": dense}


def _quantize(form, k, n, unit):
    return {"kind": "quantize", "form": form, "k": k, "n": n, "unit": unit}


def _block(batch, tokens, heads, ffn, pos=0):
    return {"kind": "block", "batch": batch, "tokens": tokens, "heads": heads, "ffn": ffn, "pos": pos}


def listed():
    return [
        # one token through one attention projection of a 7B model: the smallest call of a serving loop
        dict(_linear(1, 4096, 4096), name="w4_decode_1x4096x4096"),
        # a batch of 16 sequences, one token each, through a GPTQ layer with act-order (integer zero-points)
        dict(_linear(16, 4096, 11008, order="act", zero="integer"), name="w4_actorder_16x4096x11008"),
        # a classifier's last layer on an odd batch in half precision: K is no multiple of the group, N none of 16
        dict(_linear(100, 2000, 1000, 64, act="f16", bias=True), name="w4_ragged_100x2000x1000_f16"),
        # a prompt of 2048 tokens through the feed-forward's first projection, GPTQ layer
        dict(_linear(2048, 4096, 11008, order="act", zero="integer"), name="w4_prompt_2048x4096x11008"),
        # adapter training on frozen INT4 weights: forward and input gradient of a batch of 512 rows
        dict(_linear(512, 4096, 11008, bias=True, backward=True), name="w4_train_512x4096x11008"),
        # 8 sequences, one token each, through a W8A8 layer: activations are quantized on the way
        dict(_int8(8, 4096, 11008), name="int8_decode_8x4096x11008"),
        # the same layer on a prompt
        dict(_int8(2048, 4096, 11008, bias=True), name="int8_prompt_2048x4096x11008"),
        # f32 activations against the block format, 32-element blocks, a small batch
        dict(_q8(32, 4096, 11008, 32), name="q8_32x4096x11008_b32"),
        # and an odd large one with 128-element blocks
        dict(_q8(1000, 4096, 4096, 128), name="q8_1000x4096x4096_b128"),
        # loading: a feed-forward matrix is quantized and laid out
        dict(_quantize("w4", 4096, 11008, 128), name="w4_quantize_4096x11008"),
        # one token through a 7B-shaped block at the end of a 2048-position cache
        dict(_block(1, 1, 32, 11008, 2047), name="block_decode_1_at_2047"),
        # eight prompts of 512 tokens through the same block
        dict(_block(8, 512, 32, 11008), name="block_prompt_8x512"),
    ]


def _spread(rng, low, high):
    """A whole number between ``low`` and ``high``, even over the logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _width(rng, low, high, steps):
    """A layer's width: a multiple of one of ``steps`` (one of them at random)."""
    step = rng.choice(steps)
    return max(step, _spread(rng, low, high) // step * step)


# multiplications of the largest listed layer: no drawn one has more
_MOST = 2048 * 4096 * 11008


def draw(rng):
    kind = rng.choices(("linear", "int8", "q8", "quantize", "block"), (9, 3, 3, 1, 3))[0]
    if kind == "quantize":
        form = rng.choice(("w4", "q8", "i8"))
        unit = rng.choice((32, 64, 128)) if form != "i8" else 0
        k = _width(rng, 512, 11008, (128,) if form == "q8" else (16, 128))
        return _quantize(form, k, _width(rng, 512, 11008, (4, 16, 64)), unit)
    if kind == "block":
        heads = rng.choice((8, 16, 24, 32))
        ffn = {8: 2816, 16: 5504, 24: 8192, 32: 11008}[heads]
        if rng.random() < 0.5:
            return _block(_spread(rng, 1, 16), 1, heads, ffn, _spread(rng, 100, 4000))
        batch = _spread(rng, 1, 8)
        return _block(batch, _spread(rng, 17, 4096 // batch if batch > 2 else 1500), heads, ffn)
    k, n = _width(rng, 512, 11008, (128,) * 3 + (16,)), _width(rng, 512, 11008, (128, 64, 16, 16, 4))
    rows = _spread(rng, 1, min(2048, _MOST // (k * n)))
    if kind == "int8":
        return _int8(rows, k, n, rng.random() < 0.5)
    if kind == "q8":
        block = rng.choice((32, 128, 0))
        k = k // 128 * 128
        return _q8(rows, k, n, block or k, rng.choice(("f32", "f32", "f32", "f16")), block == 0 and rng.random() < 0.5)
    order = rng.choice(("plain", "plain", "act"))
    group = rng.choice((32, 64, 128, 128, 128))
    if order == "act":
        k = max(128, k // 128 * 128)
    plain = order == "plain"
    backward = plain and rng.random() < 0.3
    act = "f16" if plain and not backward and rng.random() < 0.2 else "f32"
    return _linear(rows, k, n, group, order=order, zero=rng.choice(("float", "integer")), act=act,
                   bias=rng.random() < 0.4, backward=backward)


# ---- what the program holds before the call --------------------------------------------------

def _normal(gen, shape, sigma=1.0):
    t = torch.empty(shape, dtype=torch.float32, device="cuda")
    return t.normal_(0.0, sigma, generator=gen)


def _activations(gen, rows, k, act="f32"):
    """N(0, 1) with a few channels that are larger throughout, as hidden states have them."""
    x = _normal(gen, (rows, k))
    loud = torch.randperm(k, generator=gen, device="cuda")[:max(1, k // 512)]
    x[:, loud] *= 20.0
    return x.to(torch.float16) if act == "f16" else x


def _w4(gen, k, n, group, order="plain", zero="float"):
    w = _normal(gen, (k, n), 0.02)
    packed, scales, zp = ops.w4_quantize_pack(w, group)
    if zero == "integer":                     # as checkpoints hold them
        zp = zp.round().clamp_(0.0, 15.0)
    g_idx = None
    if order == "act":
        g_idx = (torch.randperm(k, generator=gen, device="cuda") // group).to(torch.int32)
    return nn.QuantizedTensor.from_packed(packed, scales, zp, k, group, g_idx)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind == "quantize":
        return {"case": case, "w": _normal(gen, (case["k"], case["n"]), 0.02)}
    if kind == "block":
        dim, batch, pos = case["heads"] * 128, case["batch"], case["pos"]
        shapes = {"q": (dim, dim), "k": (dim, dim), "v": (dim, dim), "o": (dim, dim), "gate": (dim, case["ffn"]),
                  "up": (dim, case["ffn"]), "down": (case["ffn"], dim)}
        proj = {name: nn.QLinear(_w4(gen, *shape, 128), None) for name, shape in shapes.items()}
        norms = [1.0 + _normal(gen, (dim,), 0.05) for _ in range(2)]
        state = {"case": case, "block": nn.DecoderBlockW4(proj, *norms, case["heads"]),
                 "x": _normal(gen, (batch, case["tokens"], dim))}
        if pos:
            cache = (batch, pos + 1, case["heads"], 128)
            state["k"], state["v"] = _normal(gen, cache), _normal(gen, cache)
        return state
    k, n = case["k"], case["n"]
    state = {"case": case, "x": _activations(gen, case["rows"], k, case.get("act", "f32"))}
    if kind == "q8":
        state["w"] = nn.quantize(_normal(gen, (k, n), 0.02), case["block"])
        if case["dense"]:
            state["w"].prepare()
        return state
    bias = _normal(gen, (n,), 0.01) if case["bias"] else None
    if kind == "int8":
        state["layer"] = nn.Int8Linear.from_linear(nn.Linear(_normal(gen, (k, n), 0.02), bias))
        return state
    state["layer"] = nn.QLinear(_w4(gen, k, n, case["group"], case["order"], case["zero"]), bias)
    if case["backward"]:
        state["grad"] = _normal(gen, (case["rows"], n))
    return state


# ---- the call --------------------------------------------------------------------------------

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        y = state["layer"](state["x"])
        return (y, state["layer"].backward_input(state["grad"])) if case["backward"] else y
    if kind == "int8":
        return state["layer"](state["x"])
    if kind == "q8":
        return nn.matmul(state["x"], state["w"])
    if kind == "block":
        return state["block"](state["x"], state.get("k"), state.get("v"), case["pos"])
    if case["form"] == "w4":
        q = nn.QuantizedTensor.from_f32(state["w"], case["k"], case["n"], case["unit"])
        return q.packed_tensor, q.scales_tensor, q.zp_tensor
    if case["form"] == "i8":
        layer = nn.Int8Linear.from_linear(nn.Linear(state["w"]))
        return layer.wq, layer.sw
    q = nn.quantize(state["w"], case["unit"])
    return q.buffer, nn.dequantize(q)


# ---- what it cannot do without ------------------------------------------------------------------

def _w4_bytes(k, n, group):
    groups = -(-k // group)
    return groups * group * n // 2 + 2 * 4 * groups * n


def work(case):
    kind = case["kind"]
    if kind == "quantize":
        k, n = case["k"], case["n"]
        out = {"w4": _w4_bytes(k, n, case["unit"] or 1), "i8": k * n + 4 * n,
               "q8": 2 * (k * n + 4 * (k * n // (case["unit"] or 1))) + 4 * k * n}[case["form"]]
        return {"bytes": 4 * k * n + out, "flops": 0}
    if kind == "block":
        dim, ffn, batch, tokens, pos = case["heads"] * 128, case["ffn"], case["batch"], case["tokens"], case["pos"]
        rows = batch * tokens
        mults = rows * (4 * dim * dim + 3 * dim * ffn)
        weights = 4 * _w4_bytes(dim, dim, 128) + 2 * _w4_bytes(dim, ffn, 128) + _w4_bytes(ffn, dim, 128)
        if pos:
            mults += 2 * batch * (pos + 1) * dim
            cache = 4 * 2 * batch * (pos + 1) * dim
        else:
            mults += 2 * batch * (tokens * (tokens + 1) // 2) * dim
            cache = 4 * 2 * rows * dim
        return {"bytes": weights + cache + 4 * 2 * rows * dim, "flops": 2 * mults}
    rows, k, n = case["rows"], case["k"], case["n"]
    act = 2 if case.get("act") == "f16" else 4
    moved, flops = act * rows * (k + n), 2 * rows * k * n
    if kind == "int8":
        return {"bytes": moved + k * n + 4 * n, "flops": flops}
    if kind == "q8":
        return {"bytes": moved + k * n + 4 * (k * n // case["block"]), "flops": flops}
    moved += _w4_bytes(k, n, case["group"])
    return {"bytes": moved + (act * rows * (k + n) if case["backward"] else 0), "flops": flops * (2 if case["backward"] else 1)}


def tolerance(case):
    kind = case["kind"]
    if kind == "quantize":
        return "exact"
    # about four times the distance measured between these paths and the same products in float64
    if case.get("act") == "f16":        # one rounding to f16: 2.1e-4
        return {"rel": 1e-3}
    if kind == "int8":                  # exact integer sums, three f32 roundings after them: 4.4e-8
        return {"rel": 2e-7}
    if kind == "q8":                    # activations split into two f16 or four int8 parts, f32 sums: 1.5e-7
        return {"rel": 1e-6}
    return {"rel": 1e-5}                # activations as fixed point or two f16 parts, f32 sums: 1e-7 to 4e-6
