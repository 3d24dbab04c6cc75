"""Where the numbers of tiles, rows and lanes are too large for the host's reciprocals, the kernels divide: the sizes just beyond that
line and just before it, against float64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from tfjs_amd import pyhost
    pyhost.init()
    return pyhost


def _close(got, want, size, terms):
    """A sum of `terms` products in any order is off by no more roundings than that, of what it adds up (`size`)."""
    assert np.all(np.abs(got - want) <= terms * 2.0 ** -24 * size)


@pytest.mark.parametrize("batch", [65535, 65536, 65600])
def test_tiles(hip, batch):
    rng = np.random.default_rng(batch)
    a, b = rng.uniform(-1, 1, (batch, 9, 5)).astype(np.float32), rng.uniform(-1, 1, (batch, 5, 8)).astype(np.float32)
    wide = a.astype(np.float64) @ b
    _close(hip.batch_matmul(a, b), wide, np.abs(a).astype(np.float64) @ np.abs(b), 5)


@pytest.mark.parametrize("images", [3, 5])
@pytest.mark.parametrize("c,out_c", [(4, 32), (5, 33), (68, 32)])
def test_windows(hip, images, c, out_c):
    """32768 windows to a row: (rows + 256) * 32768 is 2^32 with four images."""
    rng = np.random.default_rng(images + c)
    x = rng.uniform(-1, 1, (images, 1, 32768, c)).astype(np.float32)
    w = rng.uniform(-1, 1, (1, 3, c, out_c)).astype(np.float32)
    got = hip.fused_conv2d(x, w, pad="same")[:, 0]

    def conv(x, w):
        pad = np.zeros((images, 32770, c))
        pad[:, 1:-1] = x[:, 0]
        return sum(pad[:, j:j + 32768] @ w[0, j].astype(np.float64) for j in range(3))
    _close(got, conv(x, w), conv(np.abs(x), np.abs(w)), 3 * c)


@pytest.mark.parametrize("width", [4032, 4100])
def test_depthwise_columns(hip, width):
    """1024 channel quads: (columns * quads + 64) * quads is 2^32 at 4096 columns."""
    rng = np.random.default_rng(width)
    x = rng.uniform(-1, 1, (1, 1, width, 4096)).astype(np.float32)
    w = rng.uniform(-1, 1, (3, 3, 4096, 1)).astype(np.float32)
    got = hip.fused_depthwise_conv2d(x, w, strides=1, pad="same")[0, 0]
    pad = np.zeros((width + 2, 4096), np.float32)
    pad[1:-1] = x[0, 0]
    want, size = np.zeros((width, 4096)), np.zeros((width, 4096))
    for j in range(3):
        term = pad[j:j + width].astype(np.float64) * w[1, j, :, 0]
        want += term
        size += np.abs(term)
    _close(got, want, size, 9)
