"""kd_causal_attention / kd_causal_attention_backward (kael's causal self-attention chain,
reference src/nn/transformer.cpp:114-136, as one launch forward and two backward) on the MI355X
against the C oracle's restatement of kael's composed ops (oracle/kd_oracle.c), which the CPU tests
pin to kael's CPU path and to the mathematics.

Tolerance: the reference's f32 device tolerance 1e-4 + 1e-4 |oracle| (tests/test_cuda.cpp:40-43),
elementwise, for the output, the rows' log-sum-exp and the qkv gradient. The kernels use no atomics:
a second call gives the same bits. Shapes: C4's attention (32 x 128 tokens, 4 heads; here 4 of its
batch rows), GPT-2's 12 heads, ragged lengths (no whole block of 32), one token, and 1024 positions.
Then kael's CausalSelfAttention module on the device through the fused branch against kael's CPU
path.

kd_cached_attention (new queries against a KV cache, read in place through strides) against the
oracle's cached restatement at the same tolerance: decode (one query, 1-1024 keys, every ragged
32-key group), chunks of queries after a past, a whole prompt with no past, strided views of the
fused projection and contiguous cache tensors; then kael's module with a KV cache through the
cached branch against kael's CPU path.
"""
import numpy as np
import pytest

import kd
import support
from test_oracle_attention import (cached_module, close, inputs, module_grads, numpy_attention, oracle_attention,
                                   oracle_cached, qkv_views)

pytestmark = pytest.mark.gpu

P = support.ptr
SHAPES = [(1, 1, 1), (2, 37, 3), (4, 128, 4), (1, 200, 2), (2, 64, 12), (1, 1024, 1)]


def device_attention(kdb, qkv, dout, b, t, h):
    dqkv_in, ddout = kdb.to_device(qkv), kdb.to_device(dout)
    out, lse, dq = kdb.empty((b, t, h * 64), np.float32), kdb.empty((b, h, t), np.float32), kdb.empty(qkv.shape, np.float32)
    kdb.call("causal_attention", kd.F32, out.ptr, lse.ptr, dqkv_in.ptr, b, t, h, 64)
    kdb.call("causal_attention_backward", kd.F32, dq.ptr, ddout.ptr, dqkv_in.ptr, out.ptr, lse.ptr, b, t, h, 64)
    return out.numpy(), lse.numpy(), dq.numpy()


@pytest.mark.parametrize("shape", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
def test_attention_matches_the_oracle(kdb, oracle, shape):
    b, t, h = shape
    qkv, dout = inputs(b, t, h, 64)
    want = oracle_attention(oracle, qkv, dout, b, t, h, 64)
    got = device_attention(kdb, qkv, dout, b, t, h)
    for g, w, what in zip(got, want, ("out", "lse", "qkv.grad")):
        close(g, w.astype(np.float64), what)
    again = device_attention(kdb, qkv, dout, b, t, h)
    for g, a in zip(got, again):
        np.testing.assert_array_equal(g, a)


# More than one workgroup of 128 queries per CU: the forward's products run in bf16 pieces. Around the blocks of
# 32 keys and the tiles of 128 queries.
WIDE = [(33, 33, 8), (11, 128, 24), (22, 130, 6), (10, 257, 9), (3, 385, 22)]


@pytest.mark.parametrize("shape", WIDE, ids=["x".join(map(str, s)) for s in WIDE])
def test_attention_over_many_queries(kdb, oracle, shape):
    test_attention_matches_the_oracle(kdb, oracle, shape)


def test_values_that_pieces_cannot_hold(kdb):
    """Infinities, NaN and values near the largest: what the f32 kernel gives for each batch alone. Finite values
    differ by the rounding of the two kernels (each within 2e-6 of the mathematics at these sizes)."""
    b, t, h = 13, 300, 8
    qkv = np.random.default_rng(4).normal(size=(b, t, 3, h, 64)).astype(np.float32)
    qkv[1, 40, 1, 2, 5] = np.inf  # a key: its scores are infinite, of either sign
    qkv[2, 130, 2, 3, 7] = np.inf  # values
    qkv[3, 299, 2, 0, 1] = -np.inf
    qkv[4, 150, 0, 1, 9] = np.nan  # a query
    qkv[5, 200, 2, 4, 60] = 3.4e38  # finite, infinite as one bf16
    qkv[6, 3, 1, 7, 33] = -3e30
    dev, width = kdb.to_device(qkv), h * 64
    out, lse = kdb.empty((b, t, width), np.float32), kdb.empty((b, h, t), np.float32)
    kdb.call("causal_attention", kd.F32, out.ptr, lse.ptr, dev.ptr, b, t, h, 64)
    out, lse = out.numpy(), lse.numpy()
    for i in range(8):
        one = kdb.to_device(qkv[i])
        want, want_lse = kdb.empty((t, width), np.float32), kdb.empty((h, t), np.float32)
        kdb.call("causal_attention", kd.F32, want.ptr, want_lse.ptr, one.ptr, 1, t, h, 64)
        for got, w in ((out[i], want.numpy()), (lse[i], want_lse.numpy())):
            np.testing.assert_allclose(got, w, rtol=1e-5, atol=4e-6)


def scores_of_size(b, t, h, size):
    """Operands whose scores are `size` times a permutation of 1 / t .. 1 in each head (to f32's rounding): from about
    20 t on, one key makes up each row."""
    rng = np.random.default_rng(b + t + h)
    qkv, dout = rng.uniform(-1, 1, (b, t, 3, h, 64)), rng.uniform(-1, 1, (b, t, h * 64))
    along = rng.normal(size=(b, 1, h, 64))
    along *= np.sqrt(8 * abs(size) / (along ** 2).sum(-1, keepdims=True))
    order = rng.permuted(np.tile(np.arange(1, t + 1) / t, (b, h, 1)), axis=-1).transpose(0, 2, 1)[..., None]
    qkv[:, :, 0], qkv[:, :, 1] = along, along * order * np.sign(size)
    return qkv.astype(np.float32), dout.astype(np.float32)


def check_large_scores(kdb, qkv, dout, size):
    """Against the mathematics in float64. A score is rounded by some 3e-7 of its size, which moves P by that share of
    P (1 - P), twice with the row's sum; the row's log-sum-exp L is rounded by up to 2^-24 |L|, but by no more than
    the sum of the keys beside the largest. So a key that alone makes up its row has P = 1 at any score. The other
    sums run over the 64 features and the keys, a few roundings of 2^-24 of the running sum for each term: below 1e-5
    of the sum of magnitudes."""
    b, t, _, h, _ = qkv.shape
    got = device_attention(kdb, qkv.reshape(b, t, -1), dout, b, t, h)[2]
    assert np.isfinite(got).all()
    got = got.reshape(b, t, 3, h, 64)
    x = qkv.astype(np.float64)
    q, k, v = (x[:, :, i].transpose(0, 2, 1, 3) for i in range(3))
    go = dout.astype(np.float64).reshape(b, t, h, 64).transpose(0, 2, 1, 3)
    s = np.where(np.triu(np.ones((t, t), bool), 1), -np.inf, q @ k.transpose(0, 1, 3, 2) / 8)
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    o, rest = p @ v, 1 - p
    p_err = p * (1e-5 + 6e-7 * abs(size) * rest + np.minimum(rest, 1.2e-7 * abs(size)))
    term = p_err * (np.abs(go) @ np.abs(v).transpose(0, 1, 3, 2) + (np.abs(go) * np.abs(o)).sum(-1, keepdims=True)) / 8
    want = numpy_attention(qkv.reshape(b, t, -1), dout, b, t, h, 64)[2].reshape(b, t, 3, h, 64)
    bounds = term @ np.abs(k), term.transpose(0, 1, 3, 2) @ np.abs(q), p_err.transpose(0, 1, 3, 2) @ np.abs(go)
    for i, (bound, what) in enumerate(zip(bounds, "qkv")):
        err, bound = np.abs(got[:, :, i] - want[:, :, i]), bound.transpose(0, 2, 1, 3)
        assert (err <= bound + 1e-30).all(), (what, (err / (bound + 1e-30)).max())


@pytest.mark.parametrize("size", [10, 100, -100, 1.2e3, -1.2e4, 1.2e6, -1.2e6, 1.2e8, -1.2e9, 1.2e10, 1e12, -1e12])
@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 37, 3), (1, 300, 1), (33, 33, 8), (3, 300, 30)],
                         ids=["1x1x1", "2x37x3", "1x300x1", "33x33x8", "3x300x30"])
def test_gradients_at_large_scores(kdb, shape, size):
    """P is exactly 1 where one key makes up the row (row 0 of every sequence, one dominating key), at any score: the
    last two shapes have their products in bf16 pieces, forward and scores of the backward."""
    check_large_scores(kdb, *scores_of_size(*shape, size), size)


@pytest.mark.parametrize("q_size", [1e8, 1e13, 1e20, 1e30])
def test_gradients_where_pieces_overflow(kdb, q_size):
    """Queries of one block of 32 past what pieces hold (with small keys, so that the scores stay at 1e6) among ordinary
    ones; some values of V too. Forward and backward have to take the same blocks in f32."""
    size, (b, t, h) = 1e6, (3, 300, 30)
    qkv, dout = scores_of_size(b, t, h, size)
    qkv[1, :, 1, :10] /= np.float32(q_size)
    qkv[1, 40:70, 0, :10] *= np.float32(q_size)
    qkv[2, 200, 2, 3, 5], qkv[2, 10, 2, 4, 9] = 3e15, -2e14
    dout[2] *= np.float32(1e-3)
    check_large_scores(kdb, qkv, dout, size)


def test_attention_rejects_unsupported_shapes(kdb):
    x = kdb.to_device(np.zeros(3 * 64 * 4, np.float32))
    with pytest.raises(kd.KdError):
        kdb.call("causal_attention", kd.F64, x.ptr, x.ptr, x.ptr, 1, 1, 1, 64)
    with pytest.raises(kd.KdError):
        kdb.call("causal_attention", kd.F32, x.ptr, x.ptr, x.ptr, 1, 1, 2, 32)
    with pytest.raises(kd.KdError):
        kdb.call("causal_attention_backward", kd.F32, x.ptr, x.ptr, x.ptr, x.ptr, x.ptr, 1, 0, 1, 64)
    # missing or misaligned operands are rejected on the host, before any launch
    with pytest.raises(kd.KdError):
        kdb.call("causal_attention", kd.F32, None, x.ptr, x.ptr, 1, 1, 1, 64)
    with pytest.raises(kd.KdError):
        kdb.call("causal_attention", kd.F32, x.ptr, x.ptr, x.ptr + 4, 1, 1, 1, 64)
    with pytest.raises(kd.KdError):
        kdb.call("causal_attention_backward", kd.F32, x.ptr, None, x.ptr, x.ptr, x.ptr, 1, 1, 1, 64)


@pytest.mark.parametrize("shape", [(32, 128, 256, 4), (2, 9, 128, 2), (1, 200, 768, 12)],
                         ids=["c4_32x128x256x4", "2x9x128x2", "1x200x768x12"])
def test_module_through_the_fused_branch_on_the_device(kael_hip_fused, shape):
    """kael's CausalSelfAttention module with the attention on kd_causal_attention against kael's
    CPU path: output, input gradient and every parameter gradient."""
    cpu = module_grads(kael_hip_fused, 0, shape)
    dev = module_grads(kael_hip_fused, 1, shape)
    for got, want, what in zip(dev, cpu, ("out", "x.grad", "parameter grads")):
        close(got, want.astype(np.float64), what)


@pytest.mark.parametrize("seed", range(8))
def test_attention_random_shapes(kdb, oracle, seed):
    """Seeded random shapes (1-3 batch rows, 1-300 positions, 1-6 heads): every ragged tail of the
    32-row blocks, the forward and backward against the oracle at the device tolerance."""
    rng = np.random.default_rng(1000 + seed)
    b, t, h = int(rng.integers(1, 4)), int(rng.integers(1, 301)), int(rng.integers(1, 7))
    qkv, dout = inputs(b, t, h, 64, seed)
    want = oracle_attention(oracle, qkv, dout, b, t, h, 64)
    got = device_attention(kdb, qkv, dout, b, t, h)
    for g, w, what in zip(got, want, ("out", "lse", "qkv.grad")):
        try:
            close(g, w.astype(np.float64), what)
        except AssertionError as e:
            raise AssertionError(f"seed {seed}: {b}x{t}x{h}: {e}") from None


def device_cached(kdb, q, k, v, b, h, t, keys, arrays):
    """kd_cached_attention over device copies of the host arrays that q, k and v point into."""
    dev = {id(a): kdb.to_device(a) for a in arrays}
    def remap(view):
        ptr, strides = view
        for a in arrays:
            if a.ctypes.data <= ptr < a.ctypes.data + a.nbytes:
                return dev[id(a)].ptr + (ptr - a.ctypes.data), strides
        raise ValueError("pointer outside the given arrays")
    (qp, qs), (kp, ks), (vp, vs) = remap(q), remap(k), remap(v)
    out = kdb.empty((b, t, h * 64), np.float32)
    kdb.call("cached_attention", kd.F32, out.ptr, qp, P(qs), kp, P(ks), vp, P(vs), b, h, t, keys, 64)
    return out.numpy()


CACHED = [(1, 12, 1, 1), (1, 12, 1, 31), (1, 12, 1, 32), (1, 12, 1, 33), (1, 12, 1, 100), (1, 12, 1, 1024),
          (2, 3, 5, 37), (1, 2, 64, 64), (3, 1, 7, 300)]


@pytest.mark.parametrize("shape", CACHED, ids=["x".join(map(str, s)) for s in CACHED])
def test_cached_attention_matches_the_oracle(kdb, oracle, shape):
    """(batch, heads, new queries, keys): the queries are the last rows of a fused projection of
    `keys` positions, the keys and values its per-head views (strided) and, for the second call,
    contiguous [B, H, keys, 64] copies (kael's cache after its cat)."""
    b, h, t, keys = shape
    qkv, _ = inputs(b, keys, h, 64, seed=t + keys)
    q, _, _ = qkv_views(qkv, b, keys, h, 64, start=keys - t)
    _, k, v = qkv_views(qkv, b, keys, h, 64)
    want = oracle_cached(oracle, q, k, v, b, h, t, keys).astype(np.float64)
    got = device_cached(kdb, q, k, v, b, h, t, keys, [qkv])
    close(got, want, "cached (strided)")
    np.testing.assert_array_equal(device_cached(kdb, q, k, v, b, h, t, keys, [qkv]), got)
    x = qkv.reshape(b, keys, 3, h, 64)
    kc = np.ascontiguousarray(x[:, :, 1].transpose(0, 2, 1, 3))
    vc = np.ascontiguousarray(x[:, :, 2].transpose(0, 2, 1, 3))
    cs = np.array([h * keys * 64, keys * 64, 64], np.int64)
    got_c = device_cached(kdb, q, (kc.ctypes.data, cs), (vc.ctypes.data, cs), b, h, t, keys, [qkv, kc, vc])
    close(got_c, want, "cached (contiguous cache)")


def test_cached_attention_rejects_bad_arguments(kdb):
    x = kdb.to_device(np.zeros(3 * 64 * 8, np.float32))
    s = np.array([0, 0, 64], np.int64)
    bad = np.array([0, -1, 64], np.int64)
    args = lambda dtype, strides, t, keys, d: (dtype, x.ptr, x.ptr, P(strides), x.ptr, P(s), x.ptr, P(s), 1, 1, t,
                                               keys, d)
    for a in (args(kd.F64, s, 1, 1, 64), args(kd.F32, s, 1, 1, 32), args(kd.F32, s, 2, 1, 64),
              args(kd.F32, s, 0, 1, 64), args(kd.F32, bad, 1, 1, 64)):
        with pytest.raises(kd.KdError):
            kdb.call("cached_attention", *a)
    with pytest.raises(kd.KdError):
        kdb.call("cached_attention", kd.F32, None, x.ptr, P(s), x.ptr, P(s), x.ptr, P(s), 1, 1, 1, 1, 64)


@pytest.mark.parametrize("shape", [(1, 7, 40, 1, 768, 12), (2, 16, 48, 8, 256, 4), (1, 130, 131, 1, 128, 2)],
                         ids=["gpt2_heads_tokens", "c4_heads_chunks", "past130"])
def test_cached_module_through_the_branch_on_the_device(kael_hip_fused, shape):
    """kael's CausalSelfAttention with a KV cache (a prompt, then tokens or chunks, no gradient) with
    the attention on kd_cached_attention, against kael's CPU path with the cache."""
    cpu, _ = cached_module(kael_hip_fused, 0, shape)
    dev, _ = cached_module(kael_hip_fused, 1, shape)
    close(dev, cpu.astype(np.float64), "cached module")
