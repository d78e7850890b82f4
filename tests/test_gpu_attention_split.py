"""Attention of more than one query on the bf16 matrix cores: every f32 operand as three bf16 parts, against float64."""
import numpy as np
import pytest

import oracle

from gpu_util import dev, host, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from rumus_amd import ops as o
    return o


def _operands(b, nq, nkv, h, seed, sigma=1.0):
    rng = np.random.default_rng(seed)
    return tuple(rng.normal(0, s, (b, n, h, 128)).astype(np.float32) for n, s in ((nq, sigma), (nkv, sigma), (nkv, 1.0)))


# edges of a wave's 32 queries, a workgroup's 128 and a tile's 32 keys
@pytest.mark.parametrize("b,h,nq,nkv,causal", [
    (1, 2, 2, 2, True), (2, 1, 17, 17, True), (1, 3, 31, 63, True), (1, 2, 32, 32, True), (2, 2, 33, 65, False),
    (2, 8, 43, 43, True), (1, 2, 63, 200, True), (1, 1, 127, 127, True), (1, 2, 128, 160, False), (1, 1, 257, 300, True),
    (1, 1, 3, 1025, True)])
def test_parts_keep_f32_accuracy(ops, b, h, nq, nkv, causal):
    say(f"attention in parts b={b} h={h} nq={nq} nkv={nkv} causal={causal}")
    for sigma in (0.01, 1.0, 4.0):
        q, k, v = _operands(b, nq, nkv, h, nq + nkv, sigma)
        got = host(ops.attention(dev(q), dev(k), dev(v), causal)).astype(np.float64)
        want = oracle.attention(q, k, v, causal)
        # Roundings of 2^-24 that point anywhere, in the mean square.  A score is about sigma^2: its f32 sums, the scale and the
        # exponent's subtraction are within four of them, and the softmax passes a score's error on as a share of the output;
        # the sums of the weights and of the weighted rows grow like the root of their length, a third of one per root; a
        # weight and the division, two.  With any one of the six products of parts left out of the scores or of the output (modelled
        # in float64) the error at sigma = 1 is 1.9 times this and more from 17 keys on.
        bound = (4.0 * sigma ** 2 + 0.35 * np.sqrt(nkv) + 2.0) * 2.0 ** -24
        error = np.linalg.norm(got - want) / np.linalg.norm(want)
        say(f"    sigma {sigma}: {error:.2e} of {bound:.2e}")
        assert error <= bound


def test_operands_without_parts(ops):
    """Infinities and values that round to an infinite bf16 are multiplied in f32, other workgroups' rows as before."""
    say("attention, infinite and very large operands")
    q, k, v = _operands(1, 150, 150, 2, 5)
    plain = host(ops.attention(dev(q), dev(k), dev(v), False))
    q[:, :, 0, 7] = -np.abs(q[:, :, 0, 7]) - 0.1
    k[0, 40, 0, 7] = np.inf                                    # a score of -inf: the key has no weight
    seen = np.delete(np.arange(150), 40)
    got = host(ops.attention(dev(q), dev(k), dev(v), False))
    want = oracle.attention(q[:, :, :1], np.ascontiguousarray(k[:, seen, :1]), np.ascontiguousarray(v[:, seen, :1]), False)
    np.testing.assert_allclose(got[:, :, :1], want, rtol=1e-3, atol=2e-5)
    np.testing.assert_array_equal(got[:, :, 1], plain[:, :, 1])

    q, k, v = _operands(1, 40, 90, 1, 6)
    v[0, 80, 0, 3] = np.inf                                    # every query's dim 3, no other
    v[0, 5, 0, 9] = 3.4e38                                     # larger than any bf16
    k[0, 33, 0, 11], q[:, :, :, 11] = 3.4e38, 0.0
    got = host(ops.attention(dev(q), dev(k), dev(v), False))
    finite, kk = v.copy(), k.copy()
    finite[0, 80, 0, 3] = 0.0
    want = oracle.attention(q, kk, finite, False)
    assert np.isposinf(got[..., 3]).all()
    dims = np.delete(np.arange(128), 3)
    np.testing.assert_allclose(got[..., dims], want[..., dims], rtol=1e-3, atol=2e-5)


def test_scores_near_the_lowest_value(ops):
    """Scores of -1e32 are scores: they share the weight; and a NaN stays in its row."""
    say("attention, scores of -1e32")
    q, k, v = _operands(1, 5, 70, 1, 8)
    q[:], k[:] = 0.0, 0.0
    q[..., 0], k[..., 0] = -1e16, np.where(np.arange(70) < 69, 2e17, 1e17).reshape(1, 70, 1)
    got = host(ops.attention(dev(q), dev(k), dev(v), False))
    np.testing.assert_allclose(got, np.broadcast_to(v[:, 69:], got.shape), rtol=1e-6)
    q[0, 2, 0, 5] = np.nan
    got = host(ops.attention(dev(q), dev(k), dev(v), False))
    assert np.isnan(got[0, 2]).all() and np.isfinite(got[0, [0, 1, 3, 4]]).all()


@pytest.mark.parametrize("nq,nkv,causal", [(40, 90, False), (150, 150, False), (150, 300, True)])
def test_scores_that_leave_f32(ops, nq, nkv, causal):
    """Finite operands whose product is below the lowest f32: a score of -infinity, a key without weight."""
    say(f"attention, scores of -1e45, {nq} queries of {nkv} keys")
    for large in (1e22, 1e20, 3e37):
        q, k, v = _operands(1, nq, nkv, 2, nq + 1)
        k[..., 7] = 0.0
        q[:, :, 0, 7] = large * (1.0 + 0.3 * np.abs(q[:, :, 0, 7]))    # all bits of it in use
        k[0, [2, 33, nkv - 4], 0, 7] = -1e45 / large if large < 1e30 else -1e9
        got = host(ops.attention(dev(q), dev(k), dev(v), causal))
        k64 = k.astype(np.float64)
        score = np.einsum("bqhd,bkhd->bhqk", q.astype(np.float64), k64) / np.sqrt(128.0)
        if causal:
            score = np.where(np.arange(nkv) <= np.arange(nq)[:, None] + nkv - nq, score, -np.inf)
        weight = np.exp(score - score.max(-1, keepdims=True))
        want = np.einsum("bhqk,bkhd->bqhd", weight / weight.sum(-1, keepdims=True), v.astype(np.float64))
        assert np.isfinite(got).all()
        np.testing.assert_allclose(got, want, rtol=1e-3, atol=2e-5)


@pytest.mark.parametrize("nq,nkv", [(40, 90), (130, 200)])
def test_small_operands_keep_their_bits(ops, nq, nkv):
    """Values and weights so small that the last parts of them would have no bf16."""
    say(f"attention, small values and weights, {nq} queries of {nkv} keys")
    error = lambda got, want: np.linalg.norm(got.astype(np.float64) - want) / np.linalg.norm(want)
    for power in (-99, -104, -112, -118):
        q, k, v = _operands(1, nq, nkv, 2, nq)
        v[:, :, 0] *= np.float32(2.0 ** power)
        got = host(ops.attention(dev(q), dev(k), dev(v), False))
        want = oracle.attention(q, k, v, False)
        # a weight is up to 1 and down to 2^-15 here: sums of products of 2^(power - 15) and more, f32 down to 2^-149
        bound = 128 * 2.0 ** -24 + np.sqrt(nkv) * 2.0 ** -24 + 2.0 ** -22
        for head in (0, 1):
            e = error(got[:, :, head], want[:, :, head])
            say(f"    values of 2^{power if head == 0 else 0}: {e:.2e}")
            assert e <= bound
    # every key but the first has a weight of 2^-122 to 2^-117, and the first a value of zero
    q, k, v = _operands(1, nq, nkv, 1, nq + 1)
    q[:], k[:, :, :, 0], v[:, 0] = 0.0, -(118.0 + 0.5 * np.abs(k[:, :, :, 0]).clip(0, 4)) * np.log(2.0), 0.0
    q[..., 0] = np.sqrt(128.0)
    k[:, 0, :, 0] = 0.0
    v *= 1e15
    got = host(ops.attention(dev(q), dev(k), dev(v), False))
    e = error(got, oracle.attention(q, k, v, False))
    say(f"    weights of 2^-120: {e:.2e}")
    assert e <= 122 * 3 * 2.0 ** -24                          # the score: three roundings of about 120 in f32
