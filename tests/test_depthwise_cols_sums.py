"""The column kernel with running sums (5x5 filters, channel counts that are no multiple of four) at the edges of
its tiles: maps smaller than the filter, one row, ragged row chunks, lopsided padding, every epilogue form."""
import ctypes

import numpy as np
import pytest

from tfjs_amd import capi, pyhost as hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def orc():
    from oracle import pyoracle
    return pyoracle


def _last_kernel():
    name = ctypes.create_string_buffer(256)
    capi.load_library().tfhip_last_kernel(name, 256)
    return name.value.decode()


CASES = [
    # x shape, filter extent, stride, pad, activation, per-channel bias, rows per chunk (0: the library's choice)
    ((1, 1, 1, 4), 5, 1, "same", "relu", True, 0), ((2, 2, 3, 8), 5, 2, "same", "relu6", True, 0),
    ((1, 57, 43, 20), 5, 2, "same", "relu", True, 0), ((2, 23, 19, 64), 5, 1, "same", "relu6", True, 3),
    ((3, 23, 19, 64), 5, 1, "valid", "linear", False, 23), ((2, 24, 18, 12), 5, 2, "valid", "linear", True, 5),
    ((1, 30, 31, 12), 5, 2, [[0, 0], [3, 1], [0, 4], [0, 0]], "relu", True, 7),
    ((2, 9, 17, 7), 5, 1, "same", "sigmoid", True, 4), ((2, 9, 17, 7), 5, 2, "same", "elu", True, 0),
    ((2, 31, 29, 33), 3, 1, "same", "relu6", True, 14), ((2, 31, 29, 33), 3, 2, "same", "linear", False, 4),
    ((2, 31, 29, 34), 3, 1, "same", "relu6", True, 5), ((2, 31, 29, 6), 3, 2, "same", "relu", True, 0),
    ((2, 9, 17, 10), 5, 1, "same", "relu", True, 4), ((2, 9, 17, 10), 5, 2, "same", "elu", True, 0),
    ((1, 5, 200, 1), 3, 1, "same", "leakyrelu", True, 0), ((70, 4, 4, 5), 3, 2, "same", "relu", True, 0),
    ((2, 13, 11, 24), 5, 1, "same", "prelu", True, 0), ((2, 13, 11, 24), 5, 2, "same", "sigmoid", False, 6),
]


@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_depthwise_cols_sums(orc, case):
    xs, f, stride, pad, act, with_bias, rows = case
    hip.init()
    rng = np.random.default_rng(sum(xs) + f)
    x = rng.uniform(-1, 1, xs).astype(np.float32)
    w = rng.normal(0, 0.3, (f, f, xs[3], 1)).astype(np.float32)
    kw = dict(strides=stride, pad=pad, activation=act,
              bias=rng.uniform(-1, 1, (xs[3],)).astype(np.float32) if with_bias else None,
              prelu=rng.uniform(0, 1, (xs[3],)).astype(np.float32) if act == "prelu" else None)
    lib = capi.load_library()
    capi.check(lib.tfhip_set_tuning(b"dw_rows", rows or -1))
    try:
        got = hip.fused_depthwise_conv2d(x, w, **kw)
    finally:
        capi.check(lib.tfhip_set_tuning(b"dw_rows", -1))
    general = act not in ("linear", "relu", "relu6")
    assert _last_kernel() == "depthwise_cols_sums<%d, %d, %d, %s, false>" % (f, stride, 4 if xs[3] % 4 == 0 else (2 if xs[3] % 2 == 0 else 1),
                                                                     "true" if general else "false")
    want = orc.fused_depthwise_conv2d(x, w, **kw)
    assert got.shape == want.shape
    assert np.max(np.abs(got - want) / np.maximum(1.0, np.abs(want))) <= 1e-5


@pytest.mark.parametrize("f,c", [(3, 33), (5, 40)])
def test_large_result_is_streamed(f, c):
    # 8 MB and more: the same numbers, stored non-temporally
    hip.init()
    rng = np.random.default_rng(f)
    x = rng.uniform(-1, 1, (17, 61, 73, c)).astype(np.float32)
    w = rng.normal(0, 0.3, (f, f, c, 1)).astype(np.float32)
    got = hip.fused_depthwise_conv2d(x, w, pad="same", activation="relu")
    assert _last_kernel().endswith("false, true>")
    small = hip.fused_depthwise_conv2d(x[11:12], w, pad="same", activation="relu")
    assert _last_kernel().endswith("false, false>")
    np.testing.assert_array_equal(got[11:12].view(np.uint32), small.view(np.uint32))


@pytest.mark.parametrize("f,c", [(3, 16), (5, 20), (3, 15)])
@pytest.mark.parametrize("rows_out", [1, 3, 5, 7, 8, 9, 10, 11, 12, 13, 14, 15, 17, 23, 24, 25, 63, 65])
def test_every_remainder_of_workgroups_over_the_xcds(orc, f, c, rows_out):
    # one row per workgroup: what eight equal runs leave over goes as it comes
    hip.init()
    rng = np.random.default_rng(rows_out + c)
    x = rng.uniform(-1, 1, (1, rows_out, 13, c)).astype(np.float32)
    w = rng.normal(0, 0.3, (f, f, c, 1)).astype(np.float32)
    lib = capi.load_library()
    capi.check(lib.tfhip_set_tuning(b"dw_rows", 1))
    try:
        got = hip.fused_depthwise_conv2d(x, w, pad="same", activation="relu")
    finally:
        capi.check(lib.tfhip_set_tuning(b"dw_rows", -1))
    assert "_cols" in _last_kernel()
    want = orc.fused_depthwise_conv2d(x, w, pad="same", activation="relu")
    assert np.max(np.abs(got - want) / np.maximum(1.0, np.abs(want))) <= 1e-5


@pytest.mark.parametrize("f,stride,c", [(f, s, c) for f in (3, 5) for s in (1, 2) for c in (19, 22, 24)])
@pytest.mark.parametrize("h,w,batch", [(1, 9, 1), (2, 40, 3), (59, 7, 1), (131, 33, 2)])
def test_the_librarys_choice_of_rows(orc, f, stride, c, h, w, batch):
    # every kind of lane, from one row per map to more rows than a lane ever takes
    hip.init()
    rng = np.random.default_rng(h + c)
    x = rng.uniform(-1, 1, (batch, h, w, c)).astype(np.float32)
    flt = rng.normal(0, 0.3, (f, f, c, 1)).astype(np.float32)
    got = hip.fused_depthwise_conv2d(x, flt, strides=stride, pad="same", activation="relu")
    assert "_cols" in _last_kernel()
    want = orc.fused_depthwise_conv2d(x, flt, strides=stride, pad="same", activation="relu")
    assert np.max(np.abs(got - want) / np.maximum(1.0, np.abs(want))) <= 1e-5
