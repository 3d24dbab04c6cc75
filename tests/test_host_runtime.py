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


MODEL = """
import tempfile
from tfjs_amd import workloads
folder = tempfile.mkdtemp()
workloads.write_model(folder, workloads.mobilenet_v2_weights(seed=1), np.uint8)
model = workloads.DeviceMobileNetV2(folder, 1)
model.set_input(np.zeros((1, 224, 224, 3), np.float32))
filters = [op["w2"] for op, _ in model.plan if op["kind"] == "pwdw"]

def write(name, value):
    buf, shape = model.weights[name]
    buf.upload(np.full(shape, value, np.float32))

def predict():
    '''Whether the call was a replay; it leaves no block behind that it did not find.'''
    live, logits = pyhost.memory_info()["live"], model._logits is not None
    model.predict()
    assert pyhost.memory_info()["live"] == live + (model._logits is not None) - logits
    return model._graph is not None

def refused(message):
    live, logits = pyhost.memory_info()["live"], model._logits is not None
    try:
        model.predict()
    except capi.HipBackendError as e:
        assert message in str(e), e
        assert pyhost.memory_info()["live"] == live - logits
        return True
    return False
"""


def test_predict_launches_where_a_recording_is_refused():
    """A filter written between two calls has to be searched for Inf / NaN again, which a recording cannot do:
    the call launches, a later one records."""
    fake_hip_util.run(MODEL + """
assert not predict()
write(filters[0], 0.5)
assert not predict()
assert predict() and predict()
live = pyhost.memory_info()["live"]
model.close()
assert pyhost.memory_info()["live"] == 0
model = workloads.DeviceMobileNetV2(folder, 1)
write(filters[3], np.nan)
assert refused("Inf or NaN") and refused("Inf or NaN")
write(filters[3], 1.0)
assert not predict()
write(filters[3], np.inf)
assert refused("Inf or NaN")        # (the recording first, then the launches)
write(filters[3], 0.25)
assert not predict() and predict()
assert errors()[0] == 0, errors()
""")


def test_a_replay_rests_on_what_its_filters_hold():
    """A kernel that multiplies padding by its filter is not replayed once that holds an Inf or a NaN, and is again
    when it is finite; predict() gives such a recording up and does what its launches do."""
    fake_hip_util.run(MODEL + """
assert not predict() and predict() and predict()
before = fake.fake_hip_launches()
write(filters[0], 0.5)              # finite: searched once, then replayed as before
assert predict()
searched = fake.fake_hip_launches()
assert predict()
assert fake.fake_hip_launches() - searched == searched - before - 2
graph = model._graph
check(lib.tfhip_graph_launch(graph))
write(filters[5], np.inf)
for _ in range(2):
    assert lib.tfhip_graph_launch(graph) != 0 and b"Inf or NaN" in lib.tfhip_last_error()
write(filters[5], 2.0)
check(lib.tfhip_graph_launch(graph))
write(filters[5], np.nan)
assert refused("tfhip_fused_pointwise_depthwise") and refused("tfhip_fused_pointwise_depthwise")
write(filters[5], 2.0)
assert not predict() and predict()
assert errors()[0] == 0, errors()
""")


def test_predict_sees_exchanged_buffers_and_knobs():
    fake_hip_util.run(MODEL + """
def kernels():
    '''what the last predict() launched or replayed'''
    return [launch(i)[0] for i in range(30)]

name = filters[0]
own, shape = model.weights[name]
other, other_input = DeviceBuffer(int(np.prod(shape)) * 4), DeviceBuffer(224 * 224 * 3 * 4)
assert not predict() and predict() and predict()
tiled = kernels()
for change, undo in [(lambda: model.weights.update({name: (other, shape)}), lambda: model.weights.update({name: (own, shape)})),
                     (lambda: setattr(model, "input", other_input), lambda: setattr(model, "input", model_input)),
                     (lambda: check(lib.tfhip_set_tuning(b"tile", 3)), lambda: check(lib.tfhip_set_tuning(b"tile", -1)))]:
    model_input = model.input
    for step in (change, undo):
        step()
        assert not predict() and predict() and predict()
        assert (kernels() == tiled) == (step is undo or "tuning" not in str(change.__code__.co_names))
check(lib.tfhip_set_tuning(b"tile", -1))     # no other value: nothing to do again
assert predict()
other.free()
assert errors()[0] == 0, errors()
""")


def test_a_recording_takes_the_launches_of_its_own_thread_only():
    """While one thread records, another's launches run, its copies work, and what it frees is kept only where the
    recording names it."""
    fake_hip_util.run("""
from concurrent.futures import ThreadPoolExecutor
pyhost.init()
other = ThreadPoolExecutor(1)
ones = np.ones(64, np.float32)

def multiply(out):
    check(lib.tfhip_fused_matmul(a.ptr, a.ptr, out.ptr, 1, 1, 8, 8, 8, 0, 0, None, None, 0, None, None, 0.2))

def elsewhere():
    mine = DeviceBuffer.from_numpy(ones)
    multiply(mine)
    where = launch()
    mine.upload(ones)
    assert mine.download(np.float32, 64).tolist() == ones.tolist()
    finite = ctypes.c_int()
    check(lib.tfhip_filter_is_finite(mine.ptr, 64, ctypes.byref(finite)))      # needs a wait for the stream
    check(lib.tfhip_graph_launch(first.value))
    mine.free()
    named.free()
    assert lib.tfhip_capture_begin() != 0 and b"already open" in lib.tfhip_last_error()
    return where

def record(body):
    graph, nodes = ctypes.c_int(), ctypes.c_int()
    check(lib.tfhip_capture_begin())
    body()
    check(lib.tfhip_capture_end(ctypes.byref(graph), ctypes.byref(nodes)))
    return graph, nodes.value

a, out, named = (DeviceBuffer.from_numpy(ones) for _ in range(3))
first, nodes = record(lambda: multiply(out))
assert nodes == 1
pooled = pyhost.memory_info()["pooled_bytes"]

def body():
    multiply(named)
    assert launch()[2]
    name, device, recorded, words = other.submit(elsewhere).result()
    assert not recorded
    multiply(out)

second, nodes = record(body)
assert nodes == 2
assert pyhost.memory_info()["pooled_bytes"] == pooled + 256      # the other thread's block; the graph keeps `named`
before = fake.fake_hip_launches()
check(lib.tfhip_graph_launch(second.value))
assert fake.fake_hip_launches() - before == 2
check(lib.tfhip_graph_destroy(second.value))
assert pyhost.memory_info()["pooled_bytes"] == pooled + 512
other.shutdown()
assert errors()[0] == 0, errors()
""")


def test_the_last_kernel_is_the_calling_threads():
    """A label's format and arguments are left behind separately and put together when they are asked for: another
    thread's launch must not come in between."""
    fake_hip_util.run("""
pyhost.init()
a, out = DeviceBuffer(4096), DeviceBuffer(4096)

def last():
    name = ctypes.create_string_buffer(256)
    check(lib.tfhip_last_kernel(name, 256))
    return name.value.decode()

def copy():
    check(lib.tfhip_copy(out.ptr, a.ptr, 4096))
    seen.append(last())

seen = []
check(lib.tfhip_fused_matmul(a.ptr, a.ptr, out.ptr, 1, 1, 8, 8, 8, 0, 0, None, None, 0, None, None, 0.2))
mine = last()
assert mine.startswith("few_rows<1, 1, ")
other = threading.Thread(target=copy)
other.start()
other.join()
assert seen == ["copy_f4"] and last() == mine, (seen, last())
""")


def test_copy_threads_fit_the_cpus_of_the_process():
    """A large transfer is copied by one thread per usable CPU, four at most, and a caller that waits for the others
    on a CPU they need sleeps."""
    fake_hip_util.run("""
def tasks():
    return set(os.listdir("/proc/self/task"))

def sleeps():
    status = open("/proc/self/task/%d/status" % threading.get_native_id()).read()
    return int(status.split("voluntary_ctxt_switches:")[1].split()[0])

pyhost.init()
cpus = sorted(os.sched_getaffinity(0))
data = np.arange(16 << 20, dtype=np.uint32).view(np.uint8)
buf = DeviceBuffer(data.nbytes)
before = tasks()
if len(sys.argv) > 1:
    os.sched_setaffinity(0, cpus[:1])
buf.upload(data)
crew = tasks() - before
assert len(crew) == min(3, len(os.sched_getaffinity(0)) - 1), crew
for task in tasks():                    # everything on one CPU from here
    os.sched_setaffinity(int(task), cpus[:1])
slept = sleeps()
buf.upload(data)
if crew:
    assert sleeps() > slept
np.testing.assert_array_equal(buf.download(np.uint8, data.nbytes), data)
""", each=([], ["one cpu"]))


def test_the_pieces_of_an_upload():
    """The first piece's copy overlaps nothing: half a megabyte where one thread copies, one from 2 MB on."""
    fake_hip_util.run("""
pyhost.init()
K = 1024
data = np.arange(16 << 20, dtype=np.uint32).view(np.uint8)
buf, sizes = DeviceBuffer(data.nbytes), (ctypes.c_uint64 * 64)()
for n, want in [(600 * K, [600]), (1024 * K, [512, 512]), (1900 * K, [512, 512, 876]), (2047 * K, [512, 512, 1023]),
                (2048 * K, [1024, 1024]), (3400 * K, [1024, 1024, 1352]), (64 << 20, [1024, 1024, 2048, 4096, 8192, 16384, 16384, 16384])]:
    fake.fake_hip_copy_sizes(sizes, 64)
    check(lib.tfhip_upload(buf.ptr, 0, data.ctypes.data, n))
    count = fake.fake_hip_copy_sizes(sizes, 64)
    assert [s // K for s in sizes[:count]] == want, (n // K, [s // K for s in sizes[:count]])
    np.testing.assert_array_equal(buf.download(np.uint8, n), data[:n])
assert errors()[0] == 0, errors()
""")


def test_a_child_copies_without_its_parents_threads():
    """A forked child has none of the threads that copied for its parent: it starts its own."""
    fake_hip_util.run("""
pyhost.init()
data = np.arange(4 << 20, dtype=np.uint32).view(np.uint8)
buf = DeviceBuffer(data.nbytes)
buf.upload(data)
child = os.fork()
if child == 0:
    buf.upload(data[::-1])
    os._exit(0 if np.array_equal(buf.download(np.uint8, data.nbytes), data[::-1]) else 1)
end = time.time() + 20
while time.time() < end:
    pid, status = os.waitpid(child, os.WNOHANG)
    if pid:
        assert status == 0, status
        break
    time.sleep(0.01)
else:
    os.kill(child, 9)
    raise AssertionError("the child waits for ever")
""")


def test_shutdown_waits_for_a_transfer():
    """The staging ring is not freed under a transfer; one that waited for the ring meanwhile fails and touches
    nothing."""
    fake_hip_util.run("""
from concurrent.futures import ThreadPoolExecutor
pyhost.init()
data = np.arange(3 << 20, dtype=np.uint32)          # 12 MB: several pieces
buf, out = DeviceBuffer(data.nbytes), np.empty_like(data)
buf.upload(data)
fake.fake_hip_copy_delay(30000)
def upload():
    return lib.tfhip_upload(buf.ptr, 0, data.ctypes.data, data.nbytes), lib.tfhip_last_error()
def download():
    return lib.tfhip_download(out.ctypes.data, buf.ptr, 0, out.nbytes), lib.tfhip_last_error()
with ThreadPoolExecutor(3) as pool:
    first = pool.submit(upload)
    while not fake.fake_hip_copies_now():
        time.sleep(0.001)
    waiting = [pool.submit(upload), pool.submit(download)]
    time.sleep(0.04)
    check(lib.tfhip_shutdown())
    assert first.result()[0] == 0
    for w in waiting:       # (ahead of the shutdown or behind it)
        rc, message = w.result()
        assert rc == 0 or b"shut down" in message, (rc, message)
fake.fake_hip_copy_delay(0)
check(lib.tfhip_init(0))
fresh = DeviceBuffer.from_numpy(data)
assert np.array_equal(fresh.download(np.uint32, data.size), data)
assert errors()[0] == 0, errors()
""")


def test_plain_tensors_are_not_held_twice():
    """What need not be decoded is uploaded into its tensor; the temporary block of the rest is bounded."""
    fake_hip_util.run("""
pyhost.init()
MB = 1 << 20

def load(sizes, quantized):
    specs = [dict(name=str(i), shape=[n if quantized else n // 4], dtype="float32") for i, n in enumerate(sizes)]
    if quantized:
        for s in specs:
            s["quantization"] = dict(dtype="uint8", scale=1.0, min=0.0)
    data = np.arange(sum(sizes) // 4, dtype=np.uint32)
    before = pyhost.memory_info()["pooled_bytes"]
    loaded = pyhost.decode_weights_to_device(data, specs)
    extra = pyhost.memory_info()["pooled_bytes"] - before
    at = 0
    for n, (buf, _) in zip(sizes, loaded.values()):
        if not quantized and n >= 4 * MB:
            assert np.array_equal(buf.download(np.uint32, n // 4), data[at // 4:(at + n) // 4])
        at += n
        buf.free()
    lib.tfhip_shutdown()
    check(lib.tfhip_init(0))
    return extra

assert load([24 * MB, 4 * MB, 8 * MB + 4], False) == 0
assert load([24 * MB, 1000, 9 * MB, 4 * MB - 4, 16], False) < 5 * MB
assert 96 * MB < load([96 * MB] * 3, True) < 288 * MB
assert errors()[0] == 0, errors()
""")


def test_two_threads_search_their_own_filters():
    """A search for Inf / NaN waits for its verdict in a word that searches share: one at a time."""
    fake_hip_util.run("""
from concurrent.futures import ThreadPoolExecutor
pyhost.init()
bad = np.ones(64, np.float32)
bad[5] = np.nan
buffers = [DeviceBuffer.from_numpy(x) for x in (bad, np.ones(64, np.float32))]
fake.fake_hip_copy_delay(50000)

def finite(buf):
    answer = ctypes.c_int()
    check(lib.tfhip_filter_is_finite(buf.ptr, 64, ctypes.byref(answer)))
    return answer.value

with ThreadPoolExecutor(2) as pool:
    first = pool.submit(finite, buffers[0])
    time.sleep(0.01)
    second = pool.submit(finite, buffers[1])
    assert (first.result(), second.result()) == (0, 1)
""")


def test_which_products_the_kernel_for_few_rows_takes():
    """Both sides of every line of its rules, by the label of the kernel that is launched."""
    fake_hip_util.run("""
pyhost.init()
big = [DeviceBuffer(64 << 20) for _ in range(3)]

def label():
    name = ctypes.create_string_buffer(256)
    check(lib.tfhip_last_kernel(name, 256))
    return name.value.decode()

def product(m, n, k):
    check(lib.tfhip_fused_matmul(big[0].ptr, big[1].ptr, big[2].ptr, 1, 1, m, n, k, 0, 0, None, None, 0, None, None, 0.2))
    return label()

def windows(hw, c, f, out_c):
    check(lib.tfhip_fused_conv2d(big[0].ptr, big[1].ptr, big[2].ptr, 1, hw, hw, c, f, f, out_c, 1, 1, 1, 1, f // 2, f // 2, hw,
                                 hw, 0, None, None, 0, None, None, 0.2))
    return label()

for shape, want in {
    (1, 4096, 2048): "few_rows<1, 1", (1, 4000, 2049): "few_rows<1, 4", (1, 4096, 1024): "few_rows<1, 1",
    (1, 4097, 1024): "few_rows<1, 4", (16, 2048, 4096): "few_rows<1, 1", (16, 2048, 4097): "few_rows<1, 4",
    (17, 2304, 1536): "few_rows<2, 1", (17, 2304, 2049): "few_rows<2, 4", (32, 4096, 1536): "few_rows<2, 1",
    (32, 4096, 1537): "few_rows<2, 4", (32, 4100, 1536): "gemm_kernel<", (32, 4100, 1540): "few_rows<2, 4",
    (32, 4097, 768): "gemm_kernel<", (32, 4097, 769): "few_rows<2, 4", (32, 8192, 1536): "gemm_kernel<",
    (32, 8193, 1024): "few_rows<2, 4", (33, 64, 319): "gemm_kernel<", (33, 64, 320): "few_rows<1, 1",
    (64, 1024, 2048): "few_rows<1, 1", (64, 1024, 2049): "few_rows<1, 4", (160, 256, 8192): "few_rows<1, 4",
    (128, 768, 1536): "few_rows<2, 1", (128, 768, 1540): "gemm_kernel<", (257, 256, 320): "few_rows<2, 1",
    (513, 256, 320): "gemm_kernel<",
}.items():
    assert product(*shape).startswith(want), (shape, product(*shape), want)
for shape, want in {(14, 41, 3, 16): "gemm_kernel<", (14, 42, 3, 16): "few_rows<1, 1", (7, 256, 7, 256): "few_rows<1, 1",
                    (14, 256, 7, 256): "gemm_kernel<", (10, 256, 3, 256): "few_rows<1, 1", (10, 256, 5, 256): "gemm_kernel<",
                    (38, 256, 7, 16): "few_rows<1, 1", (28, 256, 7, 32): "gemm_kernel<", (14, 130, 5, 256): "few_rows<1, 1",
                    (20, 130, 7, 130): "gemm_kernel<"}.items():
    assert windows(*shape).startswith(want), (shape, windows(*shape), want)
# split_gemm switched off with its knob: nothing else changes; preferred: wherever it can
for value, small, large in ((-1, "few_rows<1, 1", "split_gemm<"), (99, "few_rows<1, 1", "gemm_kernel<"), (98, "split_gemm<", "split_gemm<"),
                            (80, "split_gemm<", "split_gemm<"), (3, "split_gemm<4, 3, 2", "split_gemm<4, 3, 2")):
    check(lib.tfhip_set_tuning(b"split", value))
    assert product(1, 1000, 1280).startswith(small) and product(1024, 2304, 768).startswith(large), value
    assert windows(7, 256, 7, 256).startswith(small), value
check(lib.tfhip_set_tuning(b"split", -1))
assert errors()[0] == 0, errors()
""")


def test_which_products_go_to_the_bf16_matrix_cores():
    """Both sides of the line at 0.45 GFLOP, and products of a transposed operand, on which
    gemm_kernel is faster than on others."""
    fake_hip_util.run("""
pyhost.init()
big, out = [DeviceBuffer(64 << 20) for _ in range(3)], DeviceBuffer(128 << 20)
name = ctypes.create_string_buffer(256)

def label():
    check(lib.tfhip_last_kernel(name, 256))
    return name.value.decode()

for (m, n, k), want in {(1024, 1024, 210): "gemm_kernel<", (1024, 1024, 216): "split_gemm<", (1024, 2304, 768): "split_gemm<",
                        (1024, 768, 768): "split_gemm<", (1568, 1280, 320): "split_gemm<", (933, 76, 2728): "gemm_kernel<",
                        (461, 144, 2392): "gemm_kernel<"}.items():
    check(lib.tfhip_fused_matmul(big[0].ptr, big[1].ptr, big[2].ptr, 1, 1, m, n, k, 0, 0, None, None, 0, None, None, 0.2))
    assert label().startswith(want), (m, n, k, label())
for shape, want in {(128, 384, 384, 64): "split_gemm<", (128, 512, 512, 64): "split_gemm<", (1, 1024, 3072, 768): "split_gemm<",
                    (1, 2640, 88, 2036): "gemm_kernel<", (1, 1949, 104, 1892): "gemm_kernel<", (53, 167, 164, 164): "gemm_kernel<",
                    (1, 3521, 168, 608): "gemm_kernel<"}.items():     # of a transposed operand
    check(lib.tfhip_fused_matmul(big[0].ptr, big[1].ptr, out.ptr, shape[0], *shape, 0, 1, None, None, 0, None, None, 0.2))
    assert label().startswith(want), (shape, label())
for (batch, h, w, c, f, out_c, stride), want in {(8, 56, 56, 64, 3, 64, 1): "split_gemm<", (8, 80, 34, 16, 3, 236, 2): "gemm_kernel<",
                                                 (8, 80, 34, 16, 3, 237, 2): "gemm_kernel<", (1, 19, 92, 52, 3, 236, 1): "few_rows<"}.items():
    out_h, out_w = -(-h // stride), -(-w // stride)
    pad_h, pad_w = max((out_h - 1) * stride + f - h, 0) // 2, max((out_w - 1) * stride + f - w, 0) // 2
    check(lib.tfhip_fused_conv2d(big[0].ptr, big[1].ptr, big[2].ptr, batch, h, w, c, f, f, out_c, stride, stride, 1, 1, pad_h, pad_w,
                                 out_h, out_w, 0, None, None, 0, None, None, 0.2))
    assert label().startswith(want), (batch, h, w, c, f, out_c, stride, label())
assert errors()[0] == 0, errors()
""")


def test_filters_of_many_taps_are_gathered():
    """An image of few channels under a filter that the matrix-core form does not hold: GEMM-shaped from 16 output
    channels on, however few pixels there are."""
    fake_hip_util.run("""
pyhost.init()
big = [DeviceBuffer(8 << 20) for _ in range(3)]
name = ctypes.create_string_buffer(256)
for hw, c, f, out_c, want in [(1, 3, 4, 16, "gemm_kernel<"), (16, 3, 5, 16, "gemm_kernel<"), (16, 4, 7, 64, "gemm_kernel<"),
                              (10, 4, 11, 32, "few_rows<"), (17, 3, 5, 8, "gemm_kernel<"), (16, 3, 5, 8, "conv_few_channels<8>"),
                              (16, 3, 3, 16, "conv_few_taps<"), (16, 3, 3, 8, "conv_few_channels<8>")]:
    check(lib.tfhip_fused_conv2d(big[0].ptr, big[1].ptr, big[2].ptr, 1, hw, hw, c, f, f, out_c, 1, 1, 1, 1, f // 2, f // 2, hw,
                                 hw, 0, None, None, 0, None, None, 0.2))
    check(lib.tfhip_last_kernel(name, 256))
    assert name.value.decode().startswith(want), (hw, c, f, out_c, name.value)
""")


def test_predict_replays_up_to_the_batch_where_it_pays():
    fake_hip_util.run(MODEL + """
for batch, replays in [(8, True), (9, False)]:
    model.close()
    model = workloads.DeviceMobileNetV2(folder, batch)
    model.set_input(np.zeros((batch, 224, 224, 3), np.float32))
    assert not predict() and predict() == replays and predict() == replays
""")


def test_two_threads_keep_their_partial_sums_apart():
    """Products that are cut keep their sums in one block: from the moment a launch is given it until its last kernel
    is enqueued no other launch uses or outgrows it."""
    fake_hip_util.run("""
from concurrent.futures import ThreadPoolExecutor
pyhost.init()
a, b, out = (DeviceBuffer(32 << 20) for _ in range(3))
check(lib.tfhip_set_tuning(b"splitk", 4))
fake.fake_hip_launch_delay(2000)

def product(n):      # gemm_kernel, then gemm_finish; a larger block each time
    check(lib.tfhip_fused_matmul(a.ptr, b.ptr, out.ptr, 1, 1, 1024, n, 512, 0, 0, None, None, 0, None, None, 0.2))

before = fake.fake_hip_launches()
with ThreadPoolExecutor(2) as pool:
    for done in [pool.submit(product, n) for n in (256, 1024, 2048, 3072, 512, 4096, 1536, 768)]:
        done.result()
names = [launch(i)[0] for i in reversed(range(fake.fake_hip_launches() - before))]
assert len(names) == 16
for first, second in zip(names[::2], names[1::2]):
    assert "gemm_kernel" in first and "gemm_finish" in second, names
assert errors()[0] == 0, errors()
""")


def test_slices_of_a_product_in_bf16_parts_fit_the_fixed_scratch():
    """A caller's fixed scratch (16 MiB): slices that the caller forced and that it does not hold are refused; the library's own
    choice is made among what it holds, with the tile that suits that."""
    fake_hip_util.run("""
pyhost.init()
a, b, out = (DeviceBuffer(128 << 20) for _ in range(3))

def product(m, n, k, entry=lib.tfhip_fused_matmul_noalloc):
    return entry(a.ptr, b.ptr, out.ptr, 1, 1, m, n, k, 0, 0, None, None, 0, None, None, 0.2)

check(lib.tfhip_set_tuning(b"split", 20))                 # three slices
check(product(1024, 1365, 512))                           # 12288 bytes short of the array
assert "split_gemm" in launch(1)[0] and pyhost.workspace_info()["last_splits"] == 3
launches = fake.fake_hip_launches()
assert product(1024, 1366, 512) != 0
message = lib.tfhip_last_error().decode()
assert str(3 * 1024 * 1366 * 4) in message and "16777216" in message, message
assert fake.fake_hip_launches() == launches
check(lib.tfhip_set_tuning(b"split", -1))
name = ctypes.create_string_buffer(256)

def choice(entry, *shape):
    check(product(*shape, entry))
    check(lib.tfhip_last_kernel(name, 256))
    return name.value.decode().split(",")[:3], pyhost.workspace_info()["last_splits"]

for shape, slices in (((1280, 1280, 8192), 2), ((768, 2048, 8192), 2), ((536, 1768, 13978), 3), ((1344, 1536, 8192), 1),
                      ((2432, 1024, 8192), 1)):
    tile, wanted = choice(lib.tfhip_fused_matmul, *shape)
    assert tile[0] == "split_gemm<4" and wanted * shape[0] * shape[1] * 4 > 16 << 20, (shape, tile, wanted)
    tile, taken = choice(lib.tfhip_fused_matmul_noalloc, *shape)
    assert tile[0].startswith("split_gemm<") and taken == slices, (shape, tile, taken)
assert tile == ["split_gemm<4", " 3", " 2"]               # (four slices: 128 x 128, one group)
assert errors()[0] == 0, errors()
""")


def test_a_label_is_the_symbol_that_is_launched():
    """tfhip_last_kernel names the launched kernel with its template arguments, spelled as a profiler spells them: the
    benchmark's table of measured traffic is looked up by that name."""
    fake_hip_util.run("""
from tfjs_amd.traffic import symbol
pyhost.init()
big = [DeviceBuffer(64 << 20) for _ in range(3)]
demangle = ctypes.CDLL("libstdc++.so.6").__cxa_demangle
demangle.restype = ctypes.c_char_p
label = ctypes.create_string_buffer(256)
seen = set()

def same(rc):
    check(rc)
    check(lib.tfhip_last_kernel(label, 256))
    status = ctypes.c_int()
    launched = symbol(demangle(launch()[0].split(".kd")[0].encode(), None, None, ctypes.byref(status)).decode())
    assert label.value.decode() == launched, (label.value, launched)
    seen.add(launched.split("<")[0])

def product(m, n, k, tb=0):
    same(lib.tfhip_fused_matmul(big[0].ptr, big[1].ptr, big[2].ptr, 1, 1, m, n, k, 0, tb, None, None, 0, None, None, 0.2))

def conv(hw, c, f, out_c):
    same(lib.tfhip_fused_conv2d(big[0].ptr, big[1].ptr, big[2].ptr, 1, hw, hw, c, f, f, out_c, 1, 1, 1, 1, f // 2, f // 2, hw, hw, 0,
                                None, None, 0, None, None, 0.2))

for m, n, k in ((1, 1000, 1280), (1, 4097, 1024), (16, 512, 512), (32, 768, 2304), (32, 3072, 2304), (1024, 2304, 768), (513, 256, 320),
                (100352, 16, 96), (100352, 32, 144)):
    product(m, n, k)
product(1024, 2304, 768, 1)
for shape in ((14, 64, 3, 64), (56, 64, 3, 64), (56, 21, 5, 38), (16, 3, 3, 16), (16, 3, 3, 8), (112, 21, 5, 38)):
    conv(*shape)
for n, h, w, c in ((1, 7, 7, 1280), (32, 7, 7, 1280), (64, 2, 1, 32768), (1, 7, 7, 3)):
    same(lib.tfhip_mean_hw(big[0].ptr, big[1].ptr, n, h, w, c))
for f, s in ((3, 1), (3, 2), (5, 1), (5, 2)):
    out = (57 + s - 1) // s
    same(lib.tfhip_fused_depthwise_conv2d(big[0].ptr, big[1].ptr, big[2].ptr, 1, 57, 57, 96, f, f, 1, s, s, 1, 1, f // 2, f // 2, out, out,
                                          None, None, 0, None, None, 0.2))
assert seen >= {"few_rows", "split_gemm", "gemm_kernel", "mean_hw_vec", "mean_hw", "conv_few_taps", "depthwise_3x3_cols",
                "depthwise_cols_sums"}, seen
assert errors()[0] == 0, errors()
""")


def test_choosing_the_rows_of_a_depthwise_lane_costs_the_host_little():
    """The rule that every call goes through, against a count that is given; the least of many turns."""
    fake_hip_util.run("""
pyhost.init()
a, w, out = DeviceBuffer(1 << 22), DeviceBuffer(1 << 12), DeviceBuffer(1 << 22)
pad, none = i64_array([0] * 4), None
call, best = lib.tfhip_fused_depthwise_conv2d, {}
args = [a.ptr, w.ptr, out.ptr, 1, 56, 56, 64, 3, 3, 1, 1, 1, 1, 1, 0, 0, 54, 54, none, pad, 1, none, pad, 0.2]
for turn in range(60):
    for knob in (-1, 14):
        check(lib.tfhip_set_tuning(b"dw_rows", knob))
        start = time.perf_counter()
        for _ in range(1000):
            call(*args)
        best[knob] = min(best.get(knob, 1.0), (time.perf_counter() - start) / 1000)
check(lib.tfhip_set_tuning(b"dw_rows", -1))
assert "depthwise_3x3_cols" in launch()[0]
assert best[-1] < 1.2 * best[14], best   # (1.08; with divisions 1.28)
""")


def test_the_rows_of_a_depthwise_lane_by_size():
    """Maps on which other counts measured 4 to 20% slower: many images, a result that is streamed at stride 2, channels that
    fit no float4, a handful of wavefronts."""
    fake_hip_util.run("""
pyhost.init()
a, w, out = DeviceBuffer(32 * 112 * 112 * 96 * 4), DeviceBuffer(1 << 17), DeviceBuffer(1 << 26)
zeros = i64_array([0] * 4)
for (batch, h, wd, c, stride), least, most in (((32, 112, 112, 96, 2), 4, 8), ((10, 85, 7, 80, 2), 1, 1), ((9, 44, 60, 194, 2), 3, 7), ((12, 32, 13, 929, 2), 8, 12),
                                               ((168, 23, 33, 58, 2), 6, 6), ((3, 79, 32, 357, 1), 6, 12), ((2, 89, 18, 176, 2), 1, 1)):
    oh, ow = -(-h // stride), -(-wd // stride)   # "same" padding
    top, left = max((oh - 1) * stride + 3 - h, 0) // 2, max((ow - 1) * stride + 3 - wd, 0) // 2
    check(lib.tfhip_fused_depthwise_conv2d(a.ptr, w.ptr, out.ptr, batch, h, wd, c, 3, 3, 1, stride, stride, 1, 1, top, left, oh, ow,
                                           None, zeros, 1, None, zeros, 0.2))
    vec = 4 if c % 4 == 0 else 2 if c % 2 == 0 else 1
    chunks = fake.fake_hip_grid(0) // (-(-ow * (c // vec) // 64) * batch)
    rows = -(-oh // chunks)
    assert "_cols" in launch()[0] and least <= rows <= most, ((batch, h, wd, c, stride), rows)
""")


def test_products_of_a_short_k_that_suit_the_tiled_kernel():
    """Products and windows of a few k tiles that measured 5 to 30% slower in bf16 parts (tiles of 64 x 64 or 64 x 48 that pad little,
    results of a few MB), beside others of the same extents that are faster there."""
    fake_hip_util.run("""
pyhost.init()
a, b, out = DeviceBuffer(1 << 25), DeviceBuffer(1 << 24), DeviceBuffer(1 << 27)
zeros = i64_array([0] * 4)
def name():
    text = ctypes.create_string_buffer(256)
    check(lib.tfhip_last_kernel(text, 256))
    return text.value.decode().split("<")[0]
for m, n, k, transposed, want in ((11616, 368, 14, 0, "gemm_kernel"), (32474, 112, 16, 0, "gemm_kernel"), (1280, 2032, 32, 0, "gemm_kernel"), (44122, 40, 32, 0, "gemm_kernel"),
                                  (42522, 40, 21, 0, "gemm_kernel"), (28720, 41, 27, 0, "gemm_kernel"), (46998, 33, 117, 0, "gemm_kernel"), (11558, 256, 148, 1, "gemm_kernel"),
                                  (6621, 2295, 12, 0, "split_gemm"), (1454, 4277, 23, 0, "split_gemm"), (4466, 652, 61, 0, "split_gemm"), (1613, 3645, 39, 0, "split_gemm")):
    check(lib.tfhip_fused_matmul(a.ptr, b.ptr, out.ptr, 1, 1, m, n, k, 0, transposed, None, None, 0, None, None, 0.2))
    assert name() == want, (m, n, k, transposed, name())
for (batch, h, w, c, n, f), want in (((5, 172, 122, 8, 56, 3), "gemm_kernel"), ((13, 92, 83, 8, 64, 2), "gemm_kernel"), ((8, 83, 57, 16, 112, 2), "gemm_kernel"),
                                     ((16, 67, 98, 5, 56, 2), "gemm_kernel"), ((5, 96, 85, 8, 224, 3), "split_gemm"), ((4, 92, 164, 8, 96, 2), "split_gemm"),
                                     ((5, 127, 128, 3, 101, 3), "split_gemm")):
    check(lib.tfhip_fused_conv2d(a.ptr, b.ptr, out.ptr, batch, h, w, c, f, f, n, 1, 1, 1, 1, (f - 1) // 2, (f - 1) // 2, h, w, 0, None, zeros, 0, None, zeros, 0.2))
    assert name() == want, (batch, h, w, c, n, f, name())
""")


def test_choosing_the_kernel_of_a_small_product_costs_the_host_little():
    """The estimates that a product of a few k tiles goes through, against a call that leaves them out; the least of many turns."""
    fake_hip_util.run("""
pyhost.init()
a, b, out = DeviceBuffer(1 << 20), DeviceBuffer(1 << 20), DeviceBuffer(1 << 22)
call, best = lib.tfhip_fused_matmul, {}
args = [a.ptr, b.ptr, out.ptr, 1, 1, 1500, 600, 100, 0, 0, None, None, 0, None, None, 0.2]
for turn in range(60):
    for knob in (-1, 99):
        check(lib.tfhip_set_tuning(b"split", knob))
        start = time.perf_counter()
        for _ in range(1000):
            call(*args)
        best[knob] = min(best.get(knob, 1.0), (time.perf_counter() - start) / 1000)
check(lib.tfhip_set_tuning(b"split", -1))
assert "gemm_kernel" in launch()[0]
assert best[-1] < 1.28 * best[99], best   # (1.18; with pow 1.33)
""")
