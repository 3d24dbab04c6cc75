"""Host <-> device transfers through the pinned staging ring, and the one-call weight decoder, at the sizes
where their pieces begin and end."""
import ctypes

import numpy as np
import pytest

from tfjs_amd import capi, pyhost as hip
from tfjs_amd.capi import DeviceBuffer, check, i64_array

pytestmark = pytest.mark.gpu

KB, MB = 1 << 10, 1 << 20


@pytest.mark.parametrize("nbytes", [1, 15, 512 * KB - 1, 512 * KB, 768 * KB + 3, MB, MB + 16, 4 * MB + 1, 8 * MB - 5, 8 * MB,
                                    12 * MB + 4097, 64 * MB + 1, 137 * MB + 13])
def test_upload_and_download_keep_every_byte(nbytes):
    # one piece, the short first pieces, whole slots, a ragged last one, more pieces than the ring has slots
    hip.init()
    data = np.random.default_rng(nbytes).integers(0, 256, nbytes, dtype=np.uint8)
    with DeviceBuffer(nbytes + 64) as buf:
        buf.upload(np.full(64, 7, np.uint8), nbytes)
        buf.upload(data)
        np.testing.assert_array_equal(buf.download(np.uint8, nbytes), data)
        odd = nbytes // 3
        np.testing.assert_array_equal(buf.download(np.uint8, nbytes - odd, odd), data[odd:])
        np.testing.assert_array_equal(buf.download(np.uint8, 64, nbytes), np.full(64, 7, np.uint8))


@pytest.mark.parametrize("kind", range(7))
def test_decode_spans_edges_and_alignments(kind):
    """Every kind at lengths around four elements, a wavefront's 1024 and a workgroup's 4096, at every byte
    offset: against the one-tensor decoders (or the bytes themselves), and nothing is written behind the end."""
    hip.init()
    lib = capi.load_library()
    width = [4, 1, 1, 1, 2, 2, 2][kind]
    lengths = [0, 1, 3, 4, 5, 255, 1023, 1025, 4095, 4096, 4097, 9001]
    rng = np.random.default_rng(kind)
    offsets, at = [], 0
    for i, n in enumerate(lengths * 2):
        at += 1 + i % 5                       # gaps: every alignment comes up
        offsets.append(at)
        at += n * width
    count, elems = len(offsets), lengths * 2
    raw = rng.integers(0, 256, at, dtype=np.uint8)
    outs = (ctypes.c_void_p * count)()
    scale_min = (ctypes.c_double * (2 * count))(*([0.0123, -1.5] * count))
    check(lib.tfhip_decode_weights(raw.ctypes.data, raw.size, count, i64_array(offsets), i64_array(elems),
                                   (ctypes.c_int * count)(*([kind] * count)), scale_min, outs))
    with DeviceBuffer.from_numpy(raw) as q:
        for off, n, ptr in zip(offsets, elems, outs):
            got_buf = DeviceBuffer.adopt(ptr, n * 4)
            if kind <= 1:
                if n:
                    np.testing.assert_array_equal(got_buf.download(np.uint8, n * width), raw[off:off + n * width])
            elif n:
                with DeviceBuffer(n * 4) as want:
                    if kind == 6:
                        check(lib.tfhip_dequant_f16(q.ptr + off, n, want.ptr))
                    else:
                        check(lib.tfhip_dequant_affine(q.ptr + off, 8 * width, n, 0.0123, -1.5, want.ptr, kind % 2))
                    np.testing.assert_array_equal(got_buf.download(np.uint32, n), want.download(np.uint32, n))
            got_buf.free()


def test_decode_refuses_what_lies_outside_the_buffer_and_leaves_nothing_behind():
    hip.init()
    lib = capi.load_library()
    raw = np.zeros(64, np.uint8)
    before = hip.memory_info()["live"]
    for offset, n, kind, message in [(60, 5, 2, b"outside"), (-1, 1, 2, b"outside"), (0, 33, 6, b"outside"),
                                     (0, 1, 7, b"unknown kind"), (65, 0, 2, b"outside"), (0, 1 << 50, 0, b"outside")]:
        outs = (ctypes.c_void_p * 2)()
        rc = lib.tfhip_decode_weights(raw.ctypes.data, raw.size, 2, i64_array([0, offset]), i64_array([4, n]),
                                      (ctypes.c_int * 2)(2, kind), (ctypes.c_double * 4)(1, 0, 1, 0), outs)
        assert rc != 0 and message in lib.tfhip_last_error(), lib.tfhip_last_error()
        assert hip.memory_info()["live"] == before


def test_decode_of_a_mixed_buffer_in_several_groups():
    """Plain tensors around the size that is uploaded alone, codes around them, and more codes than pass through the
    temporary block at once."""
    hip.init()
    rng = np.random.default_rng(1)
    sizes = [(4 * MB, None), (70 * MB + 1, "uint8"), (4 * MB - 4, None), (90 * MB, "uint8"), (12, None), (99 * MB + 3, "uint8"),
             (33 * MB + 1, "uint8"), (9 * MB + 4, None), (5, "uint8")]
    raw = rng.integers(0, 256, sum(n for n, _ in sizes), dtype=np.uint8)
    specs = [dict(name=str(i), dtype="float32", shape=[n if q else n // 4],
                  **(dict(quantization=dict(dtype=q, scale=0.5 + i, min=-3.0)) if q else {})) for i, (n, q) in enumerate(sizes)]
    pooled = hip.memory_info()["pooled_bytes"]
    loaded = hip.decode_weights_to_device(raw, specs)
    assert hip.memory_info()["pooled_bytes"] - pooled <= 288 * MB
    at = 0
    for i, (n, q) in enumerate(sizes):
        buf, _ = loaded[str(i)]
        codes = raw[at:at + n]
        want = (codes.astype(np.float64) * (0.5 + i) - 3.0).astype(np.float32) if q else codes.copy().view(np.float32)
        np.testing.assert_array_equal(buf.download(np.uint32, want.size), want.view(np.uint32))
        at += n
        buf.free()
