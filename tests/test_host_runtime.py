"""The library's host code on a stand-in for the HIP runtime: what one GPU cannot show (several devices) and what
must not be tried on one (memory of a device that is not the current one, a free under a running copy)."""
import fake_hip_util


def test_every_device_has_counters_of_its_own():
    """A product whose k is cut names counters; after a shutdown and an init on another device they are that
    device's, as its scratch is, and no launch names memory of another device."""
    fake_hip_util.run("""
for device in (0, 1, 0):
    check(lib.tfhip_init(device))
    bufs = [DeviceBuffer(4 * n) for n in (4095, 4095 * 64, 64)]
    for entry in (lib.tfhip_fused_matmul, lib.tfhip_fused_matmul_noalloc):
        check(entry(bufs[0].ptr, bufs[1].ptr, bufs[2].ptr, 1, 1, 1, 64, 4095, 0, 0, None, None, 0, None, None, 0.2))
        name, on, recorded, words = launch()
        assert "few_rows" in name and on == device, (name, on)
        owners = [fake.fake_hip_device_of(ctypes.c_void_p(w)) for w in words[:8]]
        named = [o for o in owners if o >= 0]
        assert len(named) == 5, owners          # a, b, c, the slices' scratch and the counters
        assert set(named) == {device}, owners
    check(lib.tfhip_shutdown())
assert errors()[0] == 0, errors()
""")
