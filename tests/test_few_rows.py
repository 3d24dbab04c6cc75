"""Small products against the oracle, at the edges of the kernel that takes them: row blocks of 16 and 32, strips of 16 and
64 columns, k groups of 16 and their slices, extents that no float4 fits, operands at odd addresses, and the
two forms of adding the slices (a counter per strip; in a recording, a launch of its own)."""
import ctypes

import numpy as np
import pytest

from tfjs_amd import capi
from tfjs_amd.capi import DeviceBuffer, check, i64_array

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    from tfjs_amd import pyhost
    pyhost.init()
    return capi.load_library()


def _last_kernel(lib):
    name = ctypes.create_string_buffer(256)
    lib.tfhip_last_kernel(name, 256)
    return name.value.decode()


class _Product:
    """out = act(a b + bias) with every operand `shift` floats into its block."""

    def __init__(self, lib, m, n, k, act, shift=0):
        rng = np.random.default_rng(m * 31 + n * 7 + k)
        self.lib, self.act, self.shift, self.shape = lib, act, shift, (m, n, k)
        self.host = [rng.uniform(-1, 1, s).astype(np.float32) for s in ((m, k), (k, n), (n,))]
        self.bufs = [DeviceBuffer.from_numpy(np.concatenate([np.full(shift, np.nan, np.float32), x.reshape(-1)])) for x in self.host]
        self.bufs.append(DeviceBuffer.from_numpy(np.full(shift + m * n, np.nan, np.float32)))

    def launch(self):
        m, n, k = self.shape
        a, b, bias, out = (buf.ptr + 4 * self.shift for buf in self.bufs)
        check(self.lib.tfhip_fused_matmul(a, b, out, 1, 1, m, n, k, 0, 0, bias, i64_array([0, 0, 1]),
                                          capi.ACTIVATIONS[self.act], None, i64_array([0] * 3), 0.2))

    def result(self):
        m, n, _ = self.shape
        return self.bufs[-1].download(np.float32, m * n, 4 * self.shift).reshape(m, n)

    def free(self):
        for buf in self.bufs:
            buf.free()


@pytest.mark.parametrize("m,n,k,act,shift", [
    (1, 1, 1, "linear", 0), (16, 16, 16, "relu", 0), (17, 17, 17, "relu6", 1), (32, 1000, 1280, "linear", 0),
    (33, 77, 513, "sigmoid", 0), (64, 65, 1030, "elu", 3), (64, 1024, 320, "leakyrelu", 0), (5, 4097, 2050, "relu", 0),
    (23, 4100, 2049, "linear", 1), (100, 1009, 1535, "linear", 0), (1, 64, 4095, "elu", 0), (2, 40, 16 * 64 * 8 + 1, "linear", 2),
    (196, 96, 576, "relu", 0), (49, 163, 961, "linear", 1), (1009, 33, 321, "relu6", 0), (81, 16, 5000, "sigmoid", 0),
])
def test_against_the_oracle(lib, m, n, k, act, shift):
    from oracle import pyoracle as orc
    p = _Product(lib, m, n, k, act, shift)
    try:
        for _ in range(2):   # (the second launch finds the counters the first one left)
            p.launch()
            assert _last_kernel(lib).startswith("few_rows<")
            got = p.result()
            want = orc.fused_matmul(p.host[0], p.host[1], bias=p.host[2], activation=act, leakyrelu_alpha=0.2)
            assert np.max(np.abs(got - want) / np.maximum(1.0, np.abs(want))) <= 1e-4
    finally:
        p.free()


@pytest.mark.parametrize("m,n,k,act,shift", [
    (20, 2309, 2053, "relu", 1), (33, 770, 2050, "linear", 0), (161, 250, 8193, "relu", 3), (16, 4097, 255, "elu", 0),
    (32, 8200, 300, "linear", 1), (256, 255, 2049, "sigmoid", 0),
])
def test_strips_of_64_columns_against_the_oracle(lib, m, n, k, act, shift):
    from oracle import pyoracle as orc
    p = _Product(lib, m, n, k, act, shift)
    try:
        p.launch()
        assert _last_kernel(lib).startswith("few_rows<%d, 4, " % (1 if m <= 16 or m > 32 else 2))
        got = p.result()
        want = orc.fused_matmul(p.host[0], p.host[1], bias=p.host[2], activation=act, leakyrelu_alpha=0.2)
        assert np.max(np.abs(got - want) / np.maximum(1.0, np.abs(want))) <= 1e-4
    finally:
        p.free()


@pytest.mark.parametrize("m,n", [(1, 17), (1, 4200), (2, 16), (16, 33), (19, 18), (23, 2304), (20, 8300)])
@pytest.mark.parametrize("k", [3, 16, 128, 129, 255, 257, 384, 395, 513, 1536, 1553, 2300])
def test_every_length_of_the_way_along_k(lib, m, n, k):
    """One to more than four groups of 16 per wavefront, whole and cut: each wavefront has one or two out and goes round.
    A sum of k products and a bias, in any order, is off by at most k + 1 roundings of what it adds up."""
    p = _Product(lib, m, n, k, "linear")
    try:
        p.launch()
        assert _last_kernel(lib).startswith("few_rows<")
        a, b, bias = (x.astype(np.float64) for x in p.host)
        assert np.all(np.abs(p.result() - (a @ b + bias)) <= (k + 1) * 2.0 ** -24 * (np.abs(a) @ np.abs(b) + np.abs(bias)))
    finally:
        p.free()


@pytest.mark.parametrize("m,n,k,form", [
    (700, 333, 501, "2, 1"), (9000, 33, 401, "2, 1"), (4097, 19, 833, "2, 1"), (2081, 130, 517, "1, 4"), (64, 4095, 384, "1, 4"),
    (33, 4096, 3000, "1, 4"), (1200, 100, 2700, "1, 4"), (1030, 515, 385, "1, 4"),
    (33, 64, 316, "1, 1"), (200, 60, 16, "1, 1"), (785, 32, 192, "1, 1"), (300, 300, 300, "2, 1"),
])
def test_every_form_of_more_than_32_rows(lib, m, n, k, form):
    """Rows and columns that end inside a tile, tiles in either order, k that ends inside a group. The bound as above. (Below
    K = 320 only operands that float4s fit are taken.)"""
    p = _Product(lib, m, n, k, "linear", int(k >= 320))
    try:
        p.launch()
        assert _last_kernel(lib).startswith("few_rows<%s, " % form)
        a, b, bias = (x.astype(np.float64) for x in p.host)
        assert np.all(np.abs(p.result() - (a @ b + bias)) <= (k + 1) * 2.0 ** -24 * (np.abs(a) @ np.abs(b) + np.abs(bias)))
    finally:
        p.free()


@pytest.mark.parametrize("xs,out_c,f,stride,dil,form", [
    ((1, 14, 13, 32), 64, 3, 1, 1, "1, 1, 3"), ((2, 70, 69, 40), 8, 3, 1, 1, "2, 1, 3"),
    ((1, 56, 56, 64), 64, 3, 1, 1, "1, 4, 3"), ((1, 56, 45, 32), 64, 3, 1, 2, "1, 4, 3"),
    ((1, 50, 47, 11), 21, 5, 1, 1, "2, 1, 5"), ((3, 113, 75, 21), 38, 5, 2, 1, "1, 4, 5"), ((2, 37, 41, 23), 70, 3, 1, 2, "2, 1, 5"),
])
def test_every_form_of_windows(lib, xs, out_c, f, stride, dil, form):
    import torch

    from tfjs_amd import pyhost as hip
    rng = np.random.default_rng(sum(xs) + out_c)
    x = rng.uniform(-1, 1, xs).astype(np.float32)
    w = rng.normal(0, 0.2, (f, f, xs[3], out_c)).astype(np.float32)
    pad = dil * (f // 2)
    got = hip.fused_conv2d(x, w, strides=stride, dilations=dil, pad=[[0, 0], [pad, pad], [pad, pad], [0, 0]])
    assert _last_kernel(lib).startswith("few_rows<%s, " % form)

    def conv(x, w):
        x, w = torch.from_numpy(x.astype(np.float64)).permute(0, 3, 1, 2), torch.from_numpy(w.astype(np.float64)).permute(3, 2, 0, 1)
        return torch.nn.functional.conv2d(x, w, stride=stride, padding=pad, dilation=dil).permute(0, 2, 3, 1).numpy()
    # f * f * in_c products in any order: no more roundings than that
    assert np.all(np.abs(got - conv(x, w)) <= f * f * xs[3] * 2.0 ** -24 * conv(np.abs(x), np.abs(w)))


def test_a_recording_gives_the_same_bits(lib):
    p = _Product(lib, 19, 200, 2000, "relu")
    try:
        p.launch()
        want = p.result()
        graph, nodes = ctypes.c_int(), ctypes.c_int()
        check(lib.tfhip_capture_begin())
        p.launch()
        check(lib.tfhip_capture_end(ctypes.byref(graph), ctypes.byref(nodes)))
        assert nodes.value == 2
        for _ in range(3):
            p.bufs[-1].upload(np.full(19 * 200, np.nan, np.float32))
            check(lib.tfhip_graph_launch(graph.value))
            np.testing.assert_array_equal(p.result().view(np.uint32), want.view(np.uint32))
            p.launch()
            np.testing.assert_array_equal(p.result().view(np.uint32), want.view(np.uint32))
        check(lib.tfhip_graph_destroy(graph.value))
    finally:
        p.free()


def test_what_lies_behind_a_row_stays_out_of_it(lib):
    """A float4 at the end of a row of A reaches into the next row: its Inf and NaN must not."""
    p = _Product(lib, 4, 20, 18, "linear")
    try:
        p.host[0][2] = np.nan
        p.host[0][3] = np.inf
        p.bufs[0].upload(p.host[0])
        p.launch()
        got = p.result()
        np.testing.assert_allclose(got[:2], p.host[0][:2].astype(np.float64) @ p.host[1] + p.host[2], rtol=0, atol=1e-5)
        assert np.isnan(got[2]).all() and not np.isfinite(got[3]).any()
    finally:
        p.free()


@pytest.mark.parametrize("xs,fs,stride,dil,pad,act", [
    ((2, 9, 11, 64), (3, 3, 64, 17), 1, 1, "same", "relu6"),          # whole units
    ((1, 20, 13, 45), (3, 3, 45, 33), 2, 1, "same", "leakyrelu"),      # units that straddle the image's edges and segments
    ((3, 7, 6, 11), (7, 5, 11, 8), 1, 1, "same", "linear"),            # windows wider than the image allows
    ((1, 12, 9, 203), (2, 2, 203, 30), 1, 2, "valid", "relu"),         # dilated: a segment per tap
    ((2, 10, 10, 64), (3, 3, 64, 200), (1, 2), (2, 1), [[0, 0], [3, 1], [0, 2], [0, 0]], "sigmoid"),
    ((1, 5, 5, 1023), (3, 3, 1023, 16), 1, 1, "same", "elu"),          # a k range cut into slices
])
def test_windows_of_an_image(lib, xs, fs, stride, dil, pad, act):
    from oracle import pyoracle as orc
    from tfjs_amd import pyhost as hip
    rng = np.random.default_rng(sum(xs) + sum(fs))
    x = rng.uniform(-1, 1, xs).astype(np.float32)
    w = rng.normal(0, 0.2, fs).astype(np.float32)
    kw = dict(strides=stride, dilations=dil, pad=pad, bias=rng.uniform(-1, 1, (fs[3],)).astype(np.float32), activation=act,
              leakyrelu_alpha=0.1)
    got = hip.fused_conv2d(x, w, **kw)
    assert _last_kernel(lib).startswith("few_rows<")
    want = orc.fused_conv2d(x, w, **kw)
    assert np.max(np.abs(got - want) / np.maximum(1.0, np.abs(want))) <= 1e-4


def test_a_cut_product_after_shutdown_and_init(lib):
    from tfjs_amd import pyhost
    bits = []
    for _ in range(2):
        p = _Product(lib, 1, 64, 4095, "linear")
        p.launch()
        bits.append(p.result().view(np.uint32))
        p.free()
        pyhost.shutdown()
        pyhost.init(0)
    np.testing.assert_array_equal(bits[0], bits[1])


def test_two_threads_multiply_at_once(lib):
    """Products that are cut, on this kernel (1 x 4095 x 64, 24 x 3000 x 2100) and on the tiled one with a pass that adds the
    slices (300 x 2600 x 260): every thread gets its own, bit for bit."""
    from concurrent.futures import ThreadPoolExecutor
    sets = [[_Product(lib, m, n, k, "relu") for m, n, k in ((1, 64, 4095), (24, 2100, 3000), (300, 260, 2600))] for _ in range(2)]
    want = []
    for p in sets[0]:
        p.launch()
        want.append(p.result().view(np.uint32))

    def serve(products):
        got = []
        for i in range(30):
            p = products[i % 3]
            p.launch()
            got.append((i % 3, p.result().view(np.uint32)))
        return got

    try:
        with ThreadPoolExecutor(2) as pool:
            for done in [pool.submit(serve, products) for products in sets]:
                for i, got in done.result():
                    np.testing.assert_array_equal(got, want[i])
    finally:
        for p in sets[0] + sets[1]:
            p.free()
