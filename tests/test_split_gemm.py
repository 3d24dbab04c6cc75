"""The kernel that multiplies float32 operands in bf16 parts (split_gemm), on every tile it has: edges of tiles, of k tiles and
of the groups that share k; windows of both kinds; epilogues; operands that six partial products cannot multiply."""
import ctypes

import numpy as np
import pytest

from tfjs_amd import capi

pytestmark = pytest.mark.gpu

SHAPES = range(8)


@pytest.fixture(scope="module")
def hip():
    from tfjs_amd import pyhost
    pyhost.init()
    return pyhost


@pytest.fixture(scope="module")
def orc():
    from oracle import pyoracle
    return pyoracle


@pytest.fixture
def split():
    """Sets the tile; unset afterwards."""
    lib = capi.load_library()

    def force(shape):
        capi.check(lib.tfhip_set_tuning(b"split", shape))
    yield force
    capi.check(lib.tfhip_set_tuning(b"split", -1))


def _took_it():
    name = ctypes.create_string_buffer(256)
    capi.load_library().tfhip_last_kernel(name, 256)
    return name.value.decode().startswith("split_gemm<")


def _relative(k):
    return (k / 16 + 12) * 2.0 ** -23 + 2.0 ** -25


def _windows(x, w):
    """The convolution at stride 1 with "same" padding, in 64 bits."""
    (n, h, wd, c), (fh, fw, _, out) = x.shape, w.shape
    padded = np.zeros((n, h + fh - 1, wd + fw - 1, c))
    padded[:, (fh - 1) // 2:(fh - 1) // 2 + h, (fw - 1) // 2:(fw - 1) // 2 + wd] = x
    return sum(padded[:, i:i + h, j:j + wd].reshape(-1, c) @ w[i, j].astype(np.float64) for i in range(fh) for j in range(fw)).reshape(n, h, wd, out)


def _with_low_parts(v):
    """Its sizes, with the last eight bits of the mantissa between 0x20 and 0x7f: less than half a unit of the second bf16 part."""
    bits = np.abs(v).view(np.uint32)
    return ((bits & 0xffffff00) | (0x20 + (bits & 0xff) * 0x5f // 0xff)).view(np.float32)


def _two_parts(v):
    return (v.view(np.uint32) & 0xffffff00).view(np.float32)


def _bound(a, b, k):
    """What a result may be off, per result: one rounding of the accumulator (truncated: an ulp, 2^-23) per matrix instruction
    of 16 k and per wavefront group, eight more for the small products, the bias and the store, and 2^-25 of each product
    for the parts left out; all relative to the sum of the products' sizes."""
    return _relative(k) * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)) + 1e-37


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (33, 31, 33), (64, 64, 64), (65, 33, 257), (128, 128, 32), (129, 130, 131), (300, 97, 100),
                                   (257, 193, 320), (40, 3, 65), (31, 250, 1000)])
def test_products(hip, split, shape, m, n, k):
    rng = np.random.default_rng(m * n + k)
    a, b = rng.standard_normal((2, m, k)).astype(np.float32), rng.standard_normal((2, k, n)).astype(np.float32)
    split(shape)
    got = hip.batch_matmul(a, b)
    assert _took_it()
    assert (np.abs(got - a.astype(np.float64) @ b.astype(np.float64)) <= _bound(a, b, k)).all()


@pytest.mark.parametrize("m,n,k,taken", [(3982, 17, 8604, True), (3982, 16, 8604, False), (3982, 32, 8603, True), (2138, 17, 10681, True),
                                         (1500, 17, 10681, False), (14871, 28, 2168, True), (11137, 19, 1441, True)])
def test_a_strip_of_columns(hip, m, n, k, taken):
    """17 to 32 columns and not too few rows, by the library's own choice."""
    rng = np.random.default_rng(m * n + k)
    a, b = rng.standard_normal((1, m, k)).astype(np.float32), rng.standard_normal((1, k, n)).astype(np.float32)
    got = hip.batch_matmul(a, b)
    assert _took_it() == taken
    assert (np.abs(got - a.astype(np.float64) @ b.astype(np.float64)) <= _bound(a, b, k)).all()


@pytest.mark.parametrize("batch,m,n,k,transposed", [(1, 1613, 3645, 39, False), (1, 4282, 3818, 32, False), (49, 506, 604, 20, False), (1, 6225, 5385, 21, False),
                                                    (18, 1007, 860, 20, True), (9, 1011, 996, 88, True),
                                                    (1, 1454, 4277, 23, False), (1, 6621, 2295, 12, False), (1, 4466, 652, 61, False)])
def test_a_short_k(hip, batch, m, n, k, transposed):
    """One or a few k tiles, by the library's own choice: what lies beyond K of the only one is zero."""
    rng = np.random.default_rng(m * n + k)
    a, b = rng.standard_normal((batch, m, k)).astype(np.float32), rng.standard_normal((batch, n, k) if transposed else (batch, k, n)).astype(np.float32)
    got = hip.batch_matmul(a, b, transpose_b=transposed)
    assert _took_it()
    for i in (0, batch - 1):
        right = b[i].T if transposed else b[i]
        assert (np.abs(got[i] - a[i].astype(np.float64) @ right) <= _bound(a[i], right, k)).all()


@pytest.mark.parametrize("xs,fs", [((5, 96, 85, 8), (3, 3, 8, 224)), ((4, 71, 143, 8), (3, 3, 8, 224)), ((5, 127, 128, 3), (3, 3, 3, 101)),
                                   ((4, 92, 164, 8), (2, 2, 8, 96)), ((6, 99, 123, 12), (3, 3, 12, 144))])
def test_windows_of_a_short_k(hip, orc, xs, fs):
    """A few k tiles of windows, whole float4s and ragged, by the library's own choice."""
    rng = np.random.default_rng(sum(xs) + sum(fs))
    x, w = rng.uniform(-1, 1, xs).astype(np.float32), rng.uniform(-1, 1, fs).astype(np.float32)
    kw = dict(strides=1, dilations=1, pad="same", bias=rng.uniform(-1, 1, (fs[3],)).astype(np.float32), activation="relu6")
    got = hip.fused_conv2d(x, w, **kw)
    assert _took_it()
    k = fs[0] * fs[1] * fs[2]
    sums, sizes = _windows(x, w), _windows(np.abs(x), np.abs(w))
    want = np.clip(sums + kw["bias"].astype(np.float64), 0, 6)
    assert (np.abs(got - want) <= _relative(k) * (sizes + np.abs(kw["bias"])) + 1e-37).all()
    # positive operands whose third parts are all positive: without those of either the sums are 2^-17 too small
    x, w = _with_low_parts(x), _with_low_parts(w)
    got = hip.fused_conv2d(x, w, strides=1, dilations=1, pad="same")
    assert _took_it()
    want = _windows(x, w)
    assert (np.abs(got - want) <= _relative(k) * want).all()
    assert (_windows(_two_parts(x), w) < (1 - _relative(k)) * want).mean() > 0.9   # (what the bound is there to see)


@pytest.mark.parametrize("shape", [s + 10 * (n - 1) for s in SHAPES for n in (1, 3)])
@pytest.mark.parametrize("m,n,k", [(1, 1, 4), (33, 31, 36), (64, 64, 64), (129, 130, 132), (300, 97, 100), (70, 64, 1300), (33, 193, 2052)])
def test_a_transposed_operand(hip, split, shape, m, n, k):
    """Its rows end where the next begins: what a fetch holds of that is not multiplied, and an Inf or NaN there neither."""
    rng = np.random.default_rng(m * n + k)
    a, b = rng.standard_normal((2, m, k)).astype(np.float32), rng.standard_normal((2, n, k)).astype(np.float32)
    split(shape)
    got = hip.batch_matmul(a, b, transpose_b=True)
    assert _took_it()
    assert (np.abs(got - a.astype(np.float64) @ b.transpose(0, 2, 1).astype(np.float64)) <= _bound(a, b.transpose(0, 2, 1), k)).all()
    b[:, n // 2] = np.nan
    a[0, m // 2] = np.inf
    with np.errstate(invalid="ignore"):
        want = a.astype(np.float64) @ b.transpose(0, 2, 1).astype(np.float64)
    got = hip.batch_matmul(a, b, transpose_b=True)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(np.isinf(got), np.isinf(want))


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("slices", [2, 3, 8])
@pytest.mark.parametrize("m,n,k", [(70, 64, 1300), (33, 97, 2049)])
def test_slices_of_k(hip, split, shape, slices, m, n, k):
    rng = np.random.default_rng(slices)
    a, b = rng.standard_normal((1, m, k)).astype(np.float32), rng.standard_normal((1, k, n)).astype(np.float32)
    split(shape + 10 * (slices - 1))
    got = hip.batch_matmul(a, b)
    assert _took_it() and hip.workspace_info()["last_splits"] == slices
    assert (np.abs(got - a.astype(np.float64) @ b.astype(np.float64)) <= _bound(a, b, k)).all()


@pytest.mark.parametrize("act", ["linear", "relu", "relu6", "prelu", "leakyrelu", "sigmoid", "elu"])
@pytest.mark.parametrize("n,tile", [(64, 6), (97, 6), (64, 23), (97, 23)])   # (23: in three slices)
def test_epilogues(hip, orc, split, act, n, tile):
    rng = np.random.default_rng(n)
    a, b = rng.uniform(-1, 1, (1, 150, 90)).astype(np.float32), rng.uniform(-1, 1, (1, 90, n)).astype(np.float32)
    for bias in (rng.uniform(-1, 1, (n,)).astype(np.float32), rng.uniform(-1, 1, (150, 1)).astype(np.float32), None):
        kw = dict(bias=bias, activation=act, leakyrelu_alpha=0.3)
        if act == "prelu":
            kw["prelu"] = rng.uniform(-1, 1, (n,)).astype(np.float32)
        split(tile)
        got = hip.fused_matmul(a, b, **kw)
        want = orc.fused_matmul(a, b, **kw)
        assert np.max(np.abs(got - want)) <= 2e-5   # 90 products of at most 1 in another order, 2^-23 each


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("xs,fs,stride,dil,pad", [
    ((2, 13, 11, 8), (3, 3, 8, 24), 1, 1, "same"), ((1, 20, 21, 4), (5, 5, 4, 36), 2, 1, "same"),
    ((2, 13, 11, 5), (3, 3, 5, 7), 1, 1, "same"), ((2, 17, 3, 2), (3, 7, 2, 130), 1, 1, "same"),
    ((1, 9, 9, 12), (3, 3, 12, 20), 1, 2, "valid"), ((1, 31, 30, 6), (5, 5, 6, 16), 1, 1, [[0, 0], [3, 0], [0, 3], [0, 0]]),
    ((3, 40, 40, 33), (1, 1, 33, 23), 2, 1, "same"),
])
def test_windows(hip, orc, split, shape, xs, fs, stride, dil, pad):
    rng = np.random.default_rng(sum(xs) + sum(fs))
    x = rng.uniform(-1, 1, xs).astype(np.float32)
    w = rng.uniform(-1, 1, fs).astype(np.float32)
    kw = dict(strides=stride, dilations=dil, pad=pad, bias=rng.uniform(-1, 1, (fs[3],)).astype(np.float32), activation="relu6")
    split(shape)
    got = hip.fused_conv2d(x, w, **kw)
    assert _took_it()
    k = fs[0] * fs[1] * fs[2]
    assert np.max(np.abs(got - orc.fused_conv2d(x, w, **kw))) <= k * (k / 16 + 12) * 2.0 ** -23 + k * 2.0 ** -24


@pytest.mark.parametrize("shape", SHAPES)
def test_what_parts_cannot_multiply(hip, split, shape):
    m, n, k = 140, 136, 200
    rng = np.random.default_rng(9)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    a[3, 7], a[5, 11], a[5, 12], a[8, 199] = np.inf, np.inf, -np.inf, np.nan
    a[20, :] = 0
    a[20, 40] = np.float32(3.4028235e38)              # rounds to Inf in bf16
    b[9, 70], b[50, 71] = -np.inf, np.nan
    a[30, :] *= np.float32(1e-35)                     # last parts below the smallest bf16, results too
    b[:, 80] = np.float32(2.0)                        # with Inf in a: Inf, though the lower parts are zero
    a[40, :] = np.float32(1e-39)                      # subnormal
    split(shape)
    with np.errstate(all="ignore"):
        got = hip.batch_matmul(a[None], b[None])[0]
        assert _took_it()
        want = (a.astype(np.float64)[:, :, None] * b.astype(np.float64)[None]).sum(1).astype(np.float32)
    assert (np.isnan(got) == np.isnan(want)).all()
    inf = np.isinf(want) & (np.arange(m) != 20)[:, None]   # (row 20 may pass the largest float on the way)
    assert (got[inf] == want[inf]).all()
    fine = np.isfinite(want) & np.isfinite(got)
    assert (fine == np.isfinite(want))[np.arange(m) != 20].all()
    got, want = np.where(fine, got, 0), np.where(fine, want, 0)
    size = np.nan_to_num(np.abs(a), posinf=0, neginf=0).astype(np.float64) @ np.nan_to_num(np.abs(b), posinf=0, neginf=0).astype(np.float64)
    assert (np.abs(got.astype(np.float64) - want) <= (k * 2.0 ** -24 + 2.0 ** -20) * size + 2.0 ** -149 * k).all()
    # tiny rows keep float32's precision
    assert (np.abs(got[30] - want[30]) <= k * 2.0 ** -24 * size[30]).all()


# Exponents of the two operands: one so small that its lower parts, or all of it, lie below the smallest bf16, against an ordinary
# or a large one; both small; sums beyond what an accumulator of scaled parts holds; an operand beyond it.
SIZES = [(-120, 100), (-125, 100), (-130, 110), (-135, 120), (-149, 126), (-140, 35), (-149, 0), (-140, -5), (-60, -64), (50, 50), (110, -100),
         (126, -70)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("form", ["plain", "transposed", "windows", "ragged windows"])
def test_operands_of_every_size(hip, split, shape, form):
    """Nothing of an operand is lost, whatever the other one is. One rounding per product, as with float32 instructions, and 24 for
    what else a result passes through; a subnormal result is off by its last place, once per product at most."""
    rng = np.random.default_rng(shape)
    mantissa = 1 + 2.0 ** -14 - 2.0 ** -20   # what bf16 parts lose of it has one sign
    split(shape)
    for small, large in SIZES:
        for ea, eb in ((small, large), (large, small)):
            if form.endswith("windows"):
                c = 8 if form == "windows" else 5
                x = np.full((1, 12, 11, c), np.ldexp(mantissa, ea), np.float32)
                w = np.ldexp(rng.uniform(1, 2, (3, 3, c, 21)), eb).astype(np.float32)
                got = hip.fused_conv2d(x, w).reshape(90, 21)
                a = np.stack([x[0, i:i + 3, j:j + 3].reshape(-1) for i in range(10) for j in range(9)])
                b = w.reshape(9 * c, 21)
            else:
                a = np.full((150, 100), np.ldexp(mantissa, ea), np.float32)
                b = np.ldexp(rng.uniform(1, 2, (100, 70)), eb).astype(np.float32)
                transposed = form == "transposed"
                got = hip.batch_matmul(a[None], np.ascontiguousarray(b.T if transposed else b)[None], transpose_b=transposed)[0]
            assert _took_it()
            want = a.astype(np.float64) @ b.astype(np.float64)   # (all positive: the sum of the products' sizes too)
            k = a.shape[1]
            assert (np.abs(got - want) <= (k + 24) * 2.0 ** -24 * want + k * 2.0 ** -149).all(), (ea, eb)


@pytest.mark.parametrize("shape", [s + 10 * (n - 1) for s in SHAPES for n in (1, 2)])
@pytest.mark.parametrize("form", ["plain", "transposed", "windows", "ragged windows"])
@pytest.mark.parametrize("largest", [1.0, 1e32])   # (the largest: among sums that are kept, and of a tile that is done again)
def test_inf_and_nan(hip, split, shape, form, largest):
    """Results that an Inf or NaN enters are what IEEE arithmetic makes of them, all others what they are without."""
    rng = np.random.default_rng(shape)
    split(shape)
    if form.endswith("windows"):
        c = 8 if form == "windows" else 5
        x, w = rng.standard_normal((1, 24, 15, c)).astype(np.float32), rng.standard_normal((3, 3, c, 37)).astype(np.float32)
        x[0, 4, 4, 2], x[0, 12, 2, 1], x[0, 12, 4, 1], x[0, 20, 10, c - 1] = np.nan, np.inf, -np.inf, np.inf
        x[0, 17, 6, 0] = largest
        w[1, 1, 2, 5], w[0, 2, 1, 6], w[:, :, :, 7] = np.inf, 0, 1   # (1: all but its high part is zero)
        a = np.stack([x[0, i:i + 3, j:j + 3].reshape(-1) for i in range(22) for j in range(13)])
        b = w.reshape(9 * c, 37)
        run = lambda: hip.fused_conv2d(x, w).reshape(a.shape[0], 37)
    else:
        m, n, k = 150, 70, 132 if form == "transposed" else 131
        a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
        a[3, 0], a[9, 100], a[9, 101], a[20, 50], a[140, k - 1] = np.inf, np.inf, -np.inf, np.nan, -np.inf
        a[30], a[31, :] = 0, 2.0 ** -149
        a[40, 7] = largest
        b[:, 11], b[0, 12], b[100, 13], b[5, 14], b[k - 1, 69] = 1, 0, 2.0 ** -149, np.inf, np.nan
        args = (np.ascontiguousarray(b.T)[None], True) if form == "transposed" else (b[None], False)
        run = lambda: hip.batch_matmul(a[None], args[0], transpose_b=args[1])[0]
    got = run()
    assert _took_it()
    with np.errstate(invalid="ignore"):
        want = (a.astype(np.float64)[:, :, None] * b.astype(np.float64)[None]).sum(1)
        size = np.abs(a.astype(np.float64)[:, :, None] * b.astype(np.float64)[None]).sum(1)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(got[np.isinf(want)], want[np.isinf(want)])
    fine = np.isfinite(want)
    # one rounding per product, as with float32 instructions, and 24 for what else a result passes through
    assert (np.abs(got[fine] - want[fine]) <= (a.shape[1] + 24) * 2.0 ** -24 * size[fine] + a.shape[1] * 2.0 ** -149).all()
