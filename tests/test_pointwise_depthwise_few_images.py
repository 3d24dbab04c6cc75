"""The tiling of the pointwise + depthwise kernels on one or two images, where slices of 16 channels and single rows
are the cheapest: against the oracle, on ragged maps and strides, with the channel-sliced and the streaming kernel."""
import ctypes

import numpy as np
import pytest

from tfjs_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,h,w,cin,mid,stride,kernel", [
    (1, 14, 14, 64, 384, 1, "expand_dw_tile<1, 4, false, 1>"),
    (1, 7, 7, 160, 960, 1, "expand_dw_tile<1, 10, false, 1>"),
    (2, 13, 11, 96, 288, 2, "expand_dw_tile<2, 6, false, 1>"),
    (1, 3, 5, 64, 64, 1, "expand_dw_tile<1, 4, false, 1>"),      # fewer rows than waves
    (1, 57, 61, 24, 144, 1, "expand_dw_stream<1, 1, true, 0, 1, 4>"),
    (1, 59, 56, 16, 96, 2, "expand_dw_stream<2, 1, false, 0, 1, 4>"),
    (2, 1, 64, 24, 48, 1, "expand_dw_stream<1, 1, true, 0, 1, 4>"),   # one row
])
def test_few_images(n, h, w, cin, mid, stride, kernel):
    from oracle import pyoracle as orc
    from tfjs_amd import pyhost as hip
    hip.init()
    rng = np.random.default_rng(h * 5 + w + cin + mid)
    x = rng.uniform(-1, 1, (n, h, w, cin)).astype(np.float32)
    w1 = rng.normal(0, 0.4, (1, 1, cin, mid)).astype(np.float32)
    b1 = rng.uniform(-1, 2, (mid,)).astype(np.float32)       # positive: relu6(bias) is far from the zero padding
    w2 = rng.normal(0, 0.5, (3, 3, mid, 1)).astype(np.float32)
    b2 = rng.uniform(-1, 1, (mid,)).astype(np.float32)
    got = hip.fused_pointwise_depthwise(x, w1, w2, strides=stride, pad="same", pw_bias=b1, pw_activation="relu6",
                                        dw_bias=b2, dw_activation="relu6")
    name = ctypes.create_string_buffer(256)
    capi.load_library().tfhip_last_kernel(name, 256)
    assert name.value.decode() == kernel
    want = orc.fused_depthwise_conv2d(orc.fused_conv2d(x, w1, bias=b1, activation="relu6"), w2, strides=stride,
                                      pad="same", bias=b2, activation="relu6")
    assert np.max(np.abs(got - want) / np.maximum(1.0, np.abs(want))) <= 1e-4
