"""Where the numbers of tiles, rows and lanes are too large for the host's reciprocals, the kernels divide: the sizes just beyond that
line and just before it, against float64, each with the kernel that it is meant for."""
import ctypes

import numpy as np
import pytest

from tfjs_amd import capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from tfjs_amd import pyhost
    pyhost.init()
    return pyhost


@pytest.fixture
def tuning():
    """Sets knobs; all unset afterwards."""
    lib, names = capi.load_library(), []

    def force(name, value):
        names.append(name)
        capi.check(lib.tfhip_set_tuning(name.encode(), value))
    yield force
    for name in names:
        capi.check(lib.tfhip_set_tuning(name.encode(), -1))


def _last_kernel():
    name = ctypes.create_string_buffer(256)
    capi.load_library().tfhip_last_kernel(name, 256)
    return name.value.decode()


def _close(got, want, size, terms):
    """A sum of `terms` products in any order is off by no more roundings than that, of what it adds up (`size`)."""
    assert np.all(np.abs(got - want) <= terms * 2.0 ** -24 * size)


@pytest.mark.parametrize("batch", [65535, 65536, 65600])
@pytest.mark.parametrize("split,kernel", [(-1, "gemm_kernel<"), (7, "split_gemm<2, 1, 4, ")])
def test_tiles(hip, tuning, batch, split, kernel):
    """One tile of either kernel for each product of the batch."""
    tuning("split", split)
    rng = np.random.default_rng(batch)
    a, b = rng.uniform(-1, 1, (batch, 9, 5)).astype(np.float32), rng.uniform(-1, 1, (batch, 5, 8)).astype(np.float32)
    wide = a.astype(np.float64) @ b
    got = hip.batch_matmul(a, b)
    assert _last_kernel().startswith(kernel)
    # (terms: 24 roundings for what a result of split_gemm passes through)
    _close(got, wide, np.abs(a).astype(np.float64) @ np.abs(b), 5 if split < 0 else 5 + 24)


@pytest.mark.parametrize("images", [3, 5])
@pytest.mark.parametrize("c,out_c,split,kernel", [(4, 36, -1, "gemm_kernel<"), (5, 33, -1, "gemm_kernel<"), (68, 32, -1, "gemm_kernel<"),
                                                  (4, 36, 4, "split_gemm<4, 2, 1, "), (5, 33, 4, "split_gemm<4, 2, 1, ")])
def test_windows(hip, tuning, images, c, out_c, split, kernel):
    """32768 windows to a row: (rows + 256) * 32768 is 2^32 with four images."""
    rng = np.random.default_rng(images + c)
    x = rng.uniform(-1, 1, (images, 1, 32768, c)).astype(np.float32)
    w = rng.uniform(-1, 1, (1, 3, c, out_c)).astype(np.float32)
    tuning("split", split)
    got = hip.fused_conv2d(x, w, pad="same")[:, 0]
    assert _last_kernel().startswith(kernel)

    def conv(x, w):
        pad = np.zeros((images, 32770, c))
        pad[:, 1:-1] = x[:, 0]
        return sum(pad[:, j:j + 32768] @ w[0, j].astype(np.float64) for j in range(3))
    _close(got, conv(x, w), conv(np.abs(x), np.abs(w)), 3 * c if split < 0 else 3 * c + 24)


@pytest.mark.parametrize("width", [4032, 4100])
def test_depthwise_columns(hip, width):
    """1024 channel quads: (columns * quads + 64) * quads is 2^32 at 4096 columns."""
    rng = np.random.default_rng(width)
    x = rng.uniform(-1, 1, (1, 1, width, 4096)).astype(np.float32)
    w = rng.uniform(-1, 1, (3, 3, 4096, 1)).astype(np.float32)
    got = hip.fused_depthwise_conv2d(x, w, strides=1, pad="same")[0, 0]
    assert _last_kernel().startswith("depthwise_3x3_cols<")
    pad = np.zeros((width + 2, 4096), np.float32)
    pad[1:-1] = x[0, 0]
    want, size = np.zeros((width, 4096)), np.zeros((width, 4096))
    for j in range(3):
        term = pad[j:j + width].astype(np.float64) * w[1, j, :, 0]
        want += term
        size += np.abs(term)
    _close(got, want, size, 9)


@pytest.mark.parametrize("kernel,height", [("expand_dw_tile", 65535), ("expand_dw_tile", 65536), ("expand_dw_stream", 46340),
                                           ("expand_dw_stream", 46341)])
def test_pointwise_and_depthwise(hip, tuning, height, kernel):
    """A workgroup per row, or a wavefront per row and half of the channels: as many, times the rows, are 2^32 at 65536 and at
    46341 rows."""
    tuning("pw_dw_stream", int(kernel == "expand_dw_stream"))
    tuning("pw_dw_tile", 1)
    tuning("tile_chunks", height)
    tuning("stream_rows", 1)
    rng = np.random.default_rng(height)
    x, w1 = rng.uniform(-1, 1, (1, height, 2, 16)).astype(np.float32), rng.uniform(-1, 1, (1, 1, 16, 32)).astype(np.float32)
    w2, b1 = rng.uniform(-1, 1, (3, 3, 32, 1)).astype(np.float32), rng.uniform(-1, 1, (32,)).astype(np.float32)
    got = hip.fused_pointwise_depthwise(x, w1, w2, pw_bias=b1, pw_activation="relu", dw_activation="relu")[0]
    assert _last_kernel().startswith(kernel + "<")

    def both(x, w1, b1, w2):
        mid = np.zeros((height + 2, 4, 32))
        mid[1:-1, 1:-1] = np.maximum(x[0].astype(np.float64) @ w1[0, 0] + b1, 0)
        return sum(mid[i:i + height, j:j + 2] * w2[i, j, :, 0] for i in range(3) for j in range(3))
    _close(got, np.maximum(both(x, w1, b1, w2), 0), both(*(np.abs(t) for t in (x, w1, b1, w2))), 17 + 9)


@pytest.mark.parametrize("shape,kernel", [((1, 2, 1, 1280), "mean_hw_vec<1, int>"), ((64, 2, 1, 32764), "mean_hw_vec<4, int>"),
                                          ((64, 2, 1, 32768), "mean_hw_vec<4, long long>"), ((3, 5, 7, 32), "mean_hw_vec<1, int>"),
                                          ((33, 9, 9, 1024), "mean_hw_vec<4, int>"), ((300, 1, 3, 16384), "mean_hw_vec<4, long long>")])
def test_mean(hip, shape, kernel):
    """8192 quads of channels: their square times 64 images is 2^32."""
    x = np.random.default_rng(shape[3]).uniform(-1, 1, shape).astype(np.float32)
    got = hip.mean_hw(x)
    assert _last_kernel() == kernel
    # every element is divided and rounded, then the sum, kept in 64 bits, is
    _close(got, x.astype(np.float64).mean((1, 2)), np.abs(x).astype(np.float64).mean((1, 2)), 2)
