"""The tiled kernel's loaders for extents that no float4 fits, against the oracle: ragged rows of A and of a
transposed B, ragged columns, windows whose units straddle the image's edges and the filter's rows, on tiles
of every width; and what a 16-byte fetch picks up beyond its row must not reach the result."""
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


@pytest.fixture(scope="module")
def orc():
    from oracle import pyoracle
    return pyoracle


def _last_kernel():
    name = ctypes.create_string_buffer(256)
    capi.load_library().tfhip_last_kernel(name, 256)
    return name.value.decode()


def _close(got, want):
    assert got.shape == want.shape
    assert np.max(np.abs(got - want) / np.maximum(1.0, np.abs(want))) <= 1e-4


@pytest.mark.parametrize("batch,m,n,k,tb,act", [
    (3, 33, 31, 35, False, "relu"), (2, 64, 65, 33, True, "linear"), (5, 101, 64, 101, False, "linear"),
    (4, 97, 97, 66, True, "relu6"), (1, 700, 19, 301, False, "sigmoid"), (1, 5001, 9, 3, False, "linear"),
    (2, 1, 1, 1, False, "linear"), (1, 301, 999, 101, True, "leakyrelu"), (1, 4099, 135, 19, False, "relu"),
])
def test_ragged_products(hip, orc, batch, m, n, k, tb, act):
    rng = np.random.default_rng(m + n + k)
    a = rng.uniform(-1, 1, (batch, m, k)).astype(np.float32)
    b = rng.uniform(-1, 1, (batch, n, k) if tb else (batch, k, n)).astype(np.float32)
    kw = dict(transpose_b=tb, activation=act, bias=rng.uniform(-1, 1, (n,)).astype(np.float32), leakyrelu_alpha=0.1)
    _close(hip.fused_matmul(a, b, **kw), orc.fused_matmul(a, b, **kw))
    assert _last_kernel().startswith("gemm_kernel<")
    assert _last_kernel().split(", ")[5] == "7"


@pytest.mark.parametrize("xs,fs,stride,dil,pad", [
    ((2, 13, 11, 5), (3, 3, 5, 7), 1, 1, "same"), ((1, 20, 21, 9), (5, 5, 9, 33), 2, 1, "same"),
    ((2, 17, 3, 2), (3, 7, 2, 130), 1, 1, "same"), ((1, 9, 9, 3), (3, 3, 3, 5), 1, 2, "valid"),
    ((3, 60, 41, 3), (7, 7, 3, 64), 2, 1, "same"), ((1, 31, 30, 4), (5, 5, 4, 16), 1, 1, [[0, 0], [3, 0], [0, 3], [0, 0]]),
    ((1, 300, 70, 6), (3, 3, 6, 10), 1, 1, "same"), ((4, 40, 40, 33), (1, 1, 33, 23), 2, 1, "same"),
])
def test_ragged_windows(hip, orc, xs, fs, stride, dil, pad):
    rng = np.random.default_rng(sum(xs) + sum(fs))
    x = rng.uniform(-1, 1, xs).astype(np.float32)
    w = rng.normal(0, 0.3, fs).astype(np.float32)
    kw = dict(strides=stride, dilations=dil, pad=pad, bias=rng.uniform(-1, 1, (fs[3],)).astype(np.float32), activation="relu6")
    _close(hip.fused_conv2d(x, w, **kw), orc.fused_conv2d(x, w, **kw))
    assert _last_kernel().startswith("gemm_kernel<")


def test_neighbouring_rows_stay_apart(hip):
    rng = np.random.default_rng(1)
    a = rng.uniform(-1, 1, (2, 40, 35)).astype(np.float32)
    b = rng.uniform(-1, 1, (2, 35, 50)).astype(np.float32)
    want = a.astype(np.float64) @ b
    a[:, 7], a[1, 9] = np.nan, np.inf
    got = hip.batch_matmul(a, b)
    bad = np.zeros((2, 40), bool)
    bad[:, 7] = bad[1, 9] = True
    assert np.isfinite(got[~bad]).all() and not np.isfinite(got[bad]).any()
    np.testing.assert_allclose(got[~bad], want[~bad], rtol=0, atol=1e-4)
    # image rows: the last unit of one reaches into the next
    x = rng.uniform(-1, 1, (1, 8, 9, 3)).astype(np.float32)
    w = rng.normal(0, 0.3, (1, 3, 3, 5)).astype(np.float32)
    x[0, 4] = np.nan
    got = hip.fused_conv2d(x, w, pad="same")
    assert np.isnan(got[0, 4]).all() and np.isfinite(np.delete(got[0], 4, 0)).all()


@pytest.mark.parametrize("xs,fs,stride", [((1, 16, 16, 3), (5, 5, 3, 16), 1), ((1, 1, 1, 3), (4, 4, 3, 16), 1),
                                          ((2, 11, 9, 4), (11, 11, 4, 32), 1), ((1, 30, 31, 1), (7, 7, 1, 64), 2)])
def test_a_few_pixels_under_a_filter_of_many_taps(hip, orc, xs, fs, stride):
    rng = np.random.default_rng(sum(xs) + sum(fs))
    x = rng.uniform(-1, 1, xs).astype(np.float32)
    w = rng.normal(0, 0.2, fs).astype(np.float32)
    kw = dict(strides=stride, pad="same", bias=rng.uniform(-1, 1, (fs[3],)).astype(np.float32), activation="relu6")
    _close(hip.fused_conv2d(x, w, **kw), orc.fused_conv2d(x, w, **kw))
    assert not _last_kernel().startswith("conv_few_channels")
