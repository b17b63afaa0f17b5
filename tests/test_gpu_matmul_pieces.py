"""f32 products on the bf16 matrix cores (kd_matmul.hip's pieces family) at the edges of its tiles,
K steps and splits, against the float64 product of the same f32 operands.

Tolerance per element, from the arithmetic: every product keeps six of the nine products of the
operands' pieces (the dropped three are below 3 * 2^-27 of it), and the running sums round at most
twice per 8 of K and once per split; each rounding is at most 2^-24 of a partial sum, which is at most
sum |a||b|. The same bound covers the small tiles and the general kernel (one rounding per K).

That bound grows with K while a lost term's error averages out, so for random operands of one size the 2-norm of the
error is bounded as well: roundings of rms 2^-24 / sqrt(3) at K / 8 partial sums that grow to the result make
2^-24 sqrt(K / 48) = 3.5e-8 sqrt(K / 16) of it, and the last few and the dropped products two more. A third piece or
the product of the second pieces left out makes 1e-6 and more at any K.
"""
import ctypes

import numpy as np
import pytest

import kd

pytestmark = pytest.mark.gpu


def product(kdb, a_store, b_store, sizes, sa, sb, out_strides=None, bias=None, out_len=None):
    batches, m, k, n = sizes
    so = out_strides or (m * n, n, 1)
    da, db = kdb.to_device(a_store), kdb.to_device(b_store)
    out = kdb.to_device(np.full(out_len or batches * m * n, np.nan, np.float32))
    args = (kd.F32, da.ptr, db.ptr, out.ptr, kd.MatmulSizes(*sizes), kd.MatmulStrides(sa, sb, so))
    if bias is None:
        kdb.call("matmul_strided", *args)
    else:
        kdb.call("matmul_strided_bias", *args, kdb.to_device(bias).ptr)
    return out.numpy()


def check(got, a, b, bias=None):
    """a [.., m, k] and b [.., k, n] as the call sees them."""
    a, b = a.astype(np.float64), b.astype(np.float64)
    want, size, k = a @ b, np.abs(a) @ np.abs(b), a.shape[-1]
    if bias is not None:
        want, size = want + bias, size + np.abs(bias)
    err = np.abs(got.reshape(want.shape) - want)
    assert (err <= (k + 72) * 2.0 ** -24 * size).all(), (err / size).max() * 2 ** 24
    return np.linalg.norm(err) / np.linalg.norm(want)


# (m, k, n): around the tiles of 64, 128 and 256 and the K steps of 16 and 32, one short K step, long K
# in splits with a ragged last one, and outputs large enough for each of the tilings
SIZES = [(63, 700, 65), (65, 1001, 63), (128, 999, 129), (127, 640, 200), (17, 4099, 5), (1, 2000, 70), (200, 3000, 1),
         (700, 33, 900), (1000, 15, 1030), (999, 768, 770), (2049, 47, 2050), (4100, 40, 4000), (300, 5003, 260)]


@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("m,k,n", SIZES, ids=lambda v: str(v))
def test_ragged_products(kdb, m, k, n, layout):
    rng = np.random.default_rng(m + 7 * k + 31 * n)
    a, b = rng.normal(size=(m, k)).astype(np.float32), rng.normal(size=(k, n)).astype(np.float32)
    at, bt = layout[0] == "t", layout[1] == "t"
    bias = rng.normal(size=n).astype(np.float32) if layout == "nt" else None
    got = product(kdb, a.T.copy() if at else a, b.T.copy() if bt else b, (1, m, k, n), (0, 1, m) if at else (0, k, 1),
                  (0, 1, k) if bt else (0, n, 1), bias=bias)
    assert check(got, a, b, bias) <= 3.5e-8 * ((k / 16) ** 0.5 + 2)


@pytest.mark.parametrize("small_b", [False, True])
@pytest.mark.parametrize("k", [1, 8, 40])
@pytest.mark.parametrize("exponent", [-149, -140, -127, -126, -120, -115, -112, -110, -100, 95, 105, 111, 112, 127])
def test_operands_of_any_size_keep_their_bits(kdb, exponent, k, small_b):
    """One operand's values from the smallest subnormals to the largest, the other's such that products are near 1 (or as
    near as f32 goes): a short K, so that nothing averages out. Six products' dropped terms and a rounding per product."""
    rng = np.random.default_rng(k + 200 - exponent)
    m, n = 2000, 1030  # beyond the small tiles
    a = np.ldexp(rng.uniform(1, 2, (m, k)), exponent).astype(np.float32)  # (rounded to the subnormals' grid)
    b = np.ldexp(rng.uniform(1, 2, (k, n)), int(np.clip(-exponent, -126, 120))).astype(np.float32)
    if small_b:
        a, b, m, n = b.T.copy(), a.T.copy(), n, m
    got = product(kdb, a, b, (1, m, k, n), (0, k, 1), (0, n, 1)).reshape(m, n)
    want = a.astype(np.float64) @ b.astype(np.float64)
    assert np.isfinite(got).all()
    assert (np.abs(got - want) <= (k + 3) * 2.0 ** -24 * want + 2.0 ** -149).all()


def test_magnitudes_that_one_bf16_cannot_hold(kdb):
    """Operands whose low pieces are subnormal, and rows of very different sizes."""
    rng = np.random.default_rng(3)
    a, b = rng.normal(size=(130, 800)).astype(np.float32), rng.normal(size=(800, 90)).astype(np.float32)
    a *= (10.0 ** rng.integers(-36, 30, (130, 1))).astype(np.float32)
    b *= np.float32(1e-2)
    check(product(kdb, a, b, (1, 130, 800, 90), (0, 800, 1), (0, 90, 1)), a, b)


@pytest.mark.parametrize("k", [48, 3000])
def test_infinities_and_nan_as_an_f32_product_has_them(kdb, k):
    rng = np.random.default_rng(k)
    m, n = 300, 520
    a, b = rng.normal(size=(m, k)).astype(np.float32), rng.normal(size=(k, n)).astype(np.float32)
    # 3.4e38 rounds to infinity in bf16; its neighbours are small, so that no f32 product overflows but one
    a[:, k - 2] *= np.float32(0.1)
    b[k - 2] *= np.float32(0.1)
    a[5, 3], a[40, k - 1], a[70, 0], a[200, k - 2] = np.inf, -np.inf, np.nan, 3.4e38
    b[7, 130], b[k - 2, 519] = np.inf, 3.4e38
    with np.errstate(all="ignore"):
        want = (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32)
    got = product(kdb, a, b, (1, m, k, n), (0, k, 1), (0, n, 1)).reshape(m, n)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(got[np.isinf(want)], want[np.isinf(want)])
    plain = np.isfinite(want)
    with np.errstate(all="ignore"):
        size = np.abs(a.astype(np.float64)) @ np.abs(b.astype(np.float64))
    err = np.abs(got[plain].astype(np.float64) - want[plain])
    assert (err <= (k + 72) * 2.0 ** -24 * size[plain]).all()


@pytest.mark.parametrize("case", ["steps", "broadcast", "reversed", "output", "unaligned"])
def test_strides_that_are_no_plain_matrix(kdb, case):
    """Both strides of an operand above 1, rows that repeat, negative strides, an output of strided columns, and
    operands that start and step at odd elements."""
    rng = np.random.default_rng(11)
    m, k, n = 150, 900, 140
    store = rng.normal(size=2_000_000).astype(np.float32)
    b = rng.normal(size=(k, n)).astype(np.float32)
    sa, so, out_len, start = (0, k, 1), (0, n, 1), m * n, 0
    if case == "steps":
        sa = (0, 2 * k + 1, 2)
    elif case == "broadcast":
        sa = (0, 0, 3)
    elif case == "reversed":
        sa, start = (0, -k, -1), m * k - 1
    elif case == "output":
        so, out_len = (0, 3 * n, 3), 3 * m * n
    else:
        sa, start = (0, k + 3, 1), 1
    index = start + np.arange(m)[:, None] * sa[1] + np.arange(k)[None] * sa[2]
    da, db = kdb.to_device(store), kdb.to_device(b)
    out = kdb.to_device(np.zeros(out_len, np.float32))
    kdb.call("matmul_strided", kd.F32, ctypes.c_void_p(da.ptr + 4 * start), db.ptr, out.ptr, kd.MatmulSizes(1, m, k, n),
             kd.MatmulStrides(sa, (0, n, 1), so))
    got = out.numpy()
    if case == "output":
        assert (got.reshape(m, n, 3)[:, :, 1:] == 0).all()
        got = got.reshape(m, n, 3)[:, :, 0]
    check(got, store[index], b)


@pytest.mark.parametrize("heads,bias", [(0, False), (0, True), (3, False)])
@pytest.mark.parametrize("m,k,n", [(700, 37, 900), (129, 16, 300), (260, 5, 385)], ids=str)
def test_strides_that_only_the_general_kernel_takes(kdb, m, k, n, heads, bias):
    """Both operands backwards (negative strides, which the pieces' loads do not address) in more than two small tiles a
    CU: one batch level, two levels of heads, with and without the bias."""
    rng = np.random.default_rng(m + heads)
    batches = 12
    a, b = rng.normal(size=(batches, m, k)).astype(np.float32), rng.normal(size=(batches, k, n)).astype(np.float32)
    add = rng.normal(size=n).astype(np.float32) if bias else None
    da, db, out = kdb.to_device(a), kdb.to_device(b), kdb.empty((batches, m, n), np.float32)
    # the last element of each first matrix, from where rows and columns run backwards
    pa, pb = ctypes.c_void_p(da.ptr + 4 * (m * k - 1)), ctypes.c_void_p(db.ptr + 4 * (k * n - 1))
    outer = heads or 1
    strides = kd.MatmulStrides((outer * m * k, -k, -1), (outer * k * n, -n, -1), (outer * m * n, n, 1))
    args = (kd.F32, pa, pb, out.ptr, kd.MatmulSizes(batches, m, k, n), strides)
    if heads:
        kdb.call("matmul_strided_heads", *args, kd.MatmulHeads(heads, m * k, k * n, m * n))
    elif bias:
        kdb.call("matmul_strided_bias", *args, kdb.to_device(add).ptr)
    else:
        kdb.call("matmul_strided", *args)
    check(out.numpy(), a[:, ::-1, ::-1], b[:, ::-1, ::-1], add)


def test_split_batches_of_heads(kdb):
    """A two-level batch whose K is split: partial sums by batch and head."""
    rng = np.random.default_rng(12)
    outer, heads, m, k, n = 2, 3, 70, 2100, 66
    a, b = (rng.normal(size=(outer, heads, *s)).astype(np.float32) for s in ((m, k), (k, n)))
    da, db = kdb.to_device(a), kdb.to_device(b)
    out = kdb.empty((outer, heads, m, n), np.float32)
    sizes = kd.MatmulSizes(outer * heads, m, k, n)
    strides = kd.MatmulStrides((heads * m * k, k, 1), (heads * k * n, n, 1), (heads * m * n, n, 1))
    kdb.call("matmul_strided_heads", kd.F32, da.ptr, db.ptr, out.ptr, sizes, strides,
             kd.MatmulHeads(heads, m * k, k * n, m * n))
    check(out.numpy(), a, b)


# (batches, m, k, n): few rows (one to four columns of lanes, around K's blocks of 64), few columns, tiles of 32 and 64 that
# a batch fills in part, with short K
MANY = [(600, 1, 16, 1024), (600, 3, 63, 257), (300, 4, 65, 255), (600, 5, 8, 1030), (700, 8, 5, 513), (520, 1, 130, 300),
        (5000, 1, 64, 1), (5000, 2, 257, 3), (3000, 7, 6, 4), (600, 40, 16, 130), (600, 65, 15, 70), (900, 24, 64, 24),
        (4096, 33, 17, 9), (520, 64, 33, 64)]


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("sizes", MANY, ids=["x".join(map(str, s)) for s in MANY])
def test_many_small_batches(kdb, sizes, layout):
    batches, m, k, n = sizes
    rng = np.random.default_rng(sum(sizes))
    a, b = rng.normal(size=(batches, m, k)).astype(np.float32), rng.normal(size=(batches, k, n)).astype(np.float32)
    at, bt = layout[0] == "t", layout[1] == "t"
    bias = rng.normal(size=n).astype(np.float32) if layout == "nt" else None
    got = product(kdb, np.ascontiguousarray(a.transpose(0, 2, 1)) if at else a,
                  np.ascontiguousarray(b.transpose(0, 2, 1)) if bt else b, sizes,
                  (m * k, 1, m) if at else (m * k, k, 1), (k * n, 1, k) if bt else (k * n, n, 1), bias=bias)
    check(got, a, b, bias)


def test_few_rows_by_batch_and_head(kdb):
    """A two-level batch of one-row products against rows of one shared matrix, at odd elements."""
    rng = np.random.default_rng(5)
    outer, heads, k, n = 150, 4, 30, 700
    a, b = rng.normal(size=(outer, heads, k)).astype(np.float32), rng.normal(size=(heads, k, n + 1)).astype(np.float32)
    da, db, out = kdb.to_device(a), kdb.to_device(b), kdb.empty((outer, heads, n), np.float32)
    kdb.call("matmul_strided_heads", kd.F32, da.ptr, ctypes.c_void_p(db.ptr + 4), out.ptr, kd.MatmulSizes(outer * heads, 1, k, n),
             kd.MatmulStrides((heads * k, k, 1), (0, n + 1, 1), (heads * n, n, 1)), kd.MatmulHeads(heads, k, k * (n + 1), n))
    check(out.numpy()[:, :, None], a[:, :, None], np.broadcast_to(b[None, :, :, 1:], (outer, heads, k, n)))


# The time that such products must not exceed, us: about three times what they take, which is their traffic or the launch
# rate of their workgroups; a 64x64 tile a batch took 500, 235, 258 and 275.
@pytest.mark.parametrize("sizes,limit", [((65535, 1, 256, 1), 80), ((65535, 2, 64, 1), 120), ((4096, 1, 16, 1024), 130),
                                         ((65535, 1, 16, 16), 210)], ids=str)
def test_small_batches_pay_for_no_tile(kdb, sizes, limit):
    batches, m, k, n = sizes
    a, b = np.ones((batches, m, k), np.float32), np.ones((batches, k, n), np.float32)
    da, db, out = kdb.to_device(a), kdb.to_device(b), kdb.empty((batches, m, n), np.float32)
    events = [ctypes.c_void_p(), ctypes.c_void_p()]
    for e in events:
        kdb.call("event_create", ctypes.byref(e))
    ms, best = ctypes.c_float(), np.inf
    for _ in range(10):
        kdb.call("event_record", events[0])
        for _ in range(10):
            kdb.call("matmul", kd.F32, da.ptr, db.ptr, out.ptr, kd.MatmulSizes(*sizes))
        kdb.call("event_record", events[1])
        kdb.call("event_elapsed_ms", ctypes.byref(ms), *events)
        best = min(best, ms.value * 100)
    for e in events:
        kdb.call("event_destroy", e)
    assert (out.numpy() == k).all()
    assert best < limit


@pytest.mark.parametrize("n", [1, 3, 4])
@pytest.mark.parametrize("k", [6, 64])
def test_few_columns_over_more_batches_than_a_grid_dimension(kdb, k, n):
    """Over 65535 batches: up to 4 columns run, more are refused."""
    rng = np.random.default_rng(n)
    a, b = rng.normal(size=(65536 + 5, 2, k)).astype(np.float32), rng.normal(size=(65536 + 5, k, n)).astype(np.float32)
    sizes = (len(a), 2, k, n)
    check(product(kdb, a, b, sizes, (2 * k, k, 1), (k * n, n, 1)), a, b)
    x = kdb.to_device(a)
    strides = kd.MatmulStrides((2 * k, k, 1), (0, 5, 1), (10, 5, 1))
    assert kdb.lib.kd_matmul_strided(kd.F32, x.ptr, x.ptr, x.ptr, kd.MatmulSizes(len(a), 2, k, 5), strides) != 0


@pytest.mark.parametrize("m,k,n", [(300, 3000, 260), (64, 5000, 64)])
def test_captured_products_keep_no_workspace(kdb, m, k, n):
    """A product that runs in splits when it is called is one kernel of a captured graph, and its replays do not depend on
    what other calls do to the shared workspace between them."""
    lib = kdb.lib
    rng = np.random.default_rng(m)
    a, b = rng.normal(size=(m, k)).astype(np.float32), rng.normal(size=(k, n)).astype(np.float32)
    da, db, out = kdb.to_device(a), kdb.to_device(b), kdb.empty((m, n), np.float32)
    eager = kdb.empty((m, n), np.float32)
    sizes = kd.MatmulSizes(1, m, k, n)
    stream, graph, run, nodes = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_size_t()
    kdb.call("matmul", kd.F32, da.ptr, db.ptr, eager.ptr, sizes)  # the kernels are loaded outside the capture
    assert lib.hipStreamCreate(ctypes.byref(stream)) == 0
    lib.kd_get_stream.restype = ctypes.c_void_p
    before = ctypes.c_void_p(lib.kd_get_stream())
    kdb.synchronize()
    try:
        lib.kd_set_stream(stream)
        assert lib.hipStreamBeginCapture(stream, 1) == 0  # thread-local
        rc = lib.kd_matmul(kd.F32, da.ptr, db.ptr, out.ptr, sizes)
        assert lib.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0 and rc == 0
        assert lib.hipGraphGetNodes(graph, None, ctypes.byref(nodes)) == 0 and nodes.value == 1
        assert lib.hipGraphInstantiate(ctypes.byref(run), graph, None, None, 0) == 0
        for _ in range(3):
            kdb.call("matmul", kd.F32, da.ptr, db.ptr, eager.ptr, sizes)
            assert lib.hipGraphLaunch(run, stream) == 0
            assert lib.hipStreamSynchronize(stream) == 0
            check(out.numpy(), a, b)
            check(eager.numpy(), a, b)
    finally:
        lib.kd_set_stream(before)
        if run:
            lib.hipGraphExecDestroy(run)
        if graph:
            lib.hipGraphDestroy(graph)
        lib.hipStreamDestroy(stream)
