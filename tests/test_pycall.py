"""The compiled way into the entry points (tfjs_amd/csrc/pycall.cc) against ctypes, on a stand-in for the HIP runtime: the same
launches for every form of the arguments, the same refusals, and the general function wherever a form is not known."""
import os
import subprocess
import sys
import sysconfig

import pytest

from fake_hip_util import ROOT, run
from tfjs_amd import build, capi

BODY = """
assert capi.pycall is not None, "not built for this Python"
pyhost.init()
a, b, bias, out = (DeviceBuffer(1 << 16) for _ in range(4))
plain = ctypes.CDLL(capi.LIB_PATH)
for name in capi.pycall.NAMES:
    fn = getattr(plain, name)
    fn.argtypes, fn.restype = capi.SIGNATURES[name], ctypes.c_int
    assert getattr(lib, name).argtypes == fn.argtypes

def outcome(fn, args):
    '''what a call launches and returns, or raises (up to the argument types' names)'''
    try:
        status = fn(*args)
    except Exception as e:
        return type(e).__name__, str(e)
    return status, launch() if status == 0 else lib.tfhip_last_error()

def same(name, *args):
    got, want = outcome(getattr(lib, name), args), outcome(getattr(plain, name), args)
    assert got == want, (name, args, got, want)
    return got
"""


def test_entry_points_take_what_ctypes_takes():
    run(BODY + """
s3, s4 = i64_array([0, 0, 1]), i64_array([0, 0, 0, 1])
mm = [a.ptr, b.ptr, out.ptr, 1, 1, 8, 16, 32, 0, 0, bias.ptr, s3, 1, None, None, 0.2]
assert same("tfhip_fused_matmul", *mm)[0] == 0
for at, value in ((0, ctypes.c_void_p(a.ptr)), (3, True), (5, 0), (5, -1), (5, 1 << 62), (5, 1 << 70), (5, 8.0), (5, "8"), (5, None), (5, np.int64(8)),
                  (8, 1), (8, 1 << 40), (10, None), (10, 0), (10, -1), (11, None), (11, ctypes.cast(s3, ctypes.POINTER(ctypes.c_int64))), (11, ctypes.byref(s3)),
                  (11, (ctypes.c_int32 * 3)(0, 0, 1)), (11, [0, 0, 1]), (11, s4), (12, 99), (15, 1), (15, np.float32(0.5)), (15, float("nan")), (15, None),
                  (2, out.ptr + (1 << 16))):
    same("tfhip_fused_matmul", *(mm[:at] + [value] + mm[at + 1:]))
same("tfhip_fused_matmul", *mm[:-1])
same("tfhip_fused_matmul", *mm, 1)
same("tfhip_fused_matmul_noalloc", *mm)
cv = [a.ptr, b.ptr, out.ptr, 1, 8, 8, 4, 3, 3, 8, 1, 1, 1, 1, 1, 1, 8, 8, 0, bias.ptr, s4, 1, None, i64_array([0] * 4), 0.2]
same("tfhip_fused_conv2d", *cv)
same("tfhip_fused_conv2d_add", *cv, a.ptr)
same("tfhip_fused_depthwise_conv2d", *(cv[:9] + [1] + cv[10:18] + cv[19:]))
same("tfhip_mean_hw", a.ptr, out.ptr, 1, 7, 7, 16)
""")


CALL = "dict(a=a, b=b, out=out, batch_a=1, batch_b=1, m=8, n=16, k=32%s)"


@pytest.mark.parametrize("more", [
    "", ", bias=bias, bias_strides=[0, 0, 1], activation='relu'", ", bias=bias, bias_strides=(0, 0, 1), transpose_b=True",
    ", bias_strides=[]", ", bias=None, bias_strides=None, prelu=None, prelu_strides=None", ", activation='prelu', prelu=bias, prelu_strides=[0, 0, 1]",
    # not taken as they are: the general function
    ", transpose_a=1", ", leakyrelu_alpha=1", ", bias=bias, bias_strides=np.array([0, 0, 1])", ", activation='softmax'", ", activation=None",
    ", bias=3", ", nothing=1", ", bias=bias, bias_strides=[0, 0, 1.0]", ", activation=''.join(['re', 'lu'])", ", **{''.join(['bi', 'as']): bias}",
])
def test_device_fused_matmul_is_the_general_function(more):
    run(BODY + """
import types
source = types.FunctionType(pyhost.device_fused_matmul.__code__, pyhost.__dict__, "general", pyhost.device_fused_matmul.__defaults__)
def outcome_of(fn):
    try:
        return fn(**""" + CALL % more + """), launch()
    except Exception as e:
        return type(e).__name__, str(e).replace("general()", "device_fused_matmul()")
assert outcome_of(pyhost.device_fused_matmul) == outcome_of(source)
pyhost.device_fused_matmul(a, b, out, 1, 1, 8, 16, 32)
by_position = launch()
pyhost.device_fused_matmul(**""" + CALL % "" + """)
assert launch() == by_position
try:
    pyhost.device_fused_matmul(a, b, DeviceBuffer(4), 1, 1, 8, 16, 32)
    raise AssertionError("an output that is too small")
except capi.HipBackendError as e:
    assert "out" in str(e)
""")


DECODE = BODY + """
import types
general = types.FunctionType(pyhost.decode_weights_to_device.__code__, pyhost.__dict__, "general")

def spec(name, shape, dtype="float32", q=None, **more):
    s = dict(name=name, shape=shape, dtype=dtype)
    if q:
        s["quantization"] = dict(dtype=q, **more)
    return s

def outcome_of(fn, buffer, specs):
    '''names, shapes and sizes, and the table that the launch reads: places relative to its own, counts, scales, kinds'''
    try:
        loaded = fn(buffer, specs)
    except Exception as e:
        return type(e).__name__, str(e)
    assert all(type(buf) is DeviceBuffer for buf, _ in loaded.values())
    entries = sum(int(np.prod(s["shape"])) > 0 for s in specs)   # (an empty tensor has none)
    name, place = launch()[0], launch()[3][0]
    assert "decode_batch" in name and place or not entries
    table = [(ctypes.c_uint64 * 6).from_address(place + 48 * i) for i in range(entries)]
    outs = [buf.ptr for buf, _ in loaded.values()]
    seen = [(n, buf.nbytes, shape, type(shape)) for n, (buf, shape) in loaded.items()]
    rows = [(t[0] - place, outs.index(t[1]) if t[1] in outs else None, *t[2:]) for t in table]
    for buf, _ in loaded.values():
        buf.free()
    return seen, rows

data = np.arange(4096, dtype=np.uint8)
affine = dict(scale=0.5, min=-1)
cases = [
    [spec("a", [3, 5], "float32", "uint8", **affine), spec("b", [7], "int32", "uint16", scale=2, min=0.25), spec("c", [2, 2], "float32", "float16"),
     spec("d", [], "float32"), spec("e", [0, 4], "int32"), spec("f", [9], "bool"), spec("a2", [1], "int32", "uint8", **affine)],
    [spec("a", (3, 5), "float32", "uint8", **affine)], [spec("a", [np.int64(3)], "float32")], [spec("a", [True, 2], "float32")],
    (spec("a", [4], "float32"),), [], [spec("a", [4], "float32"), spec("a", [5], "float32")],
    [dict(spec("a", [4]), quantization=None)], [spec("a", [4], "float32", "uint8", scale=np.float64(0.5), min=0.0)],
    # refused
    [spec("a", [4], "float32", "uint8", scale=1.0)], [spec("a", [4], "int32", "float16")], [spec("a", [4], "float32", "int4", **affine)],
    [spec("a", [4], "string")], [spec("a", [4], "bool", "uint8", **affine)], [spec("a", [4096], "float32")], [spec("a", [1 << 40, 1 << 40], "float32")],
    [spec("a", [-1], "float32")], [dict(name="a", dtype="float32")], [dict(shape=[1], dtype="float32")], [None], None,
]
for specs in cases:
    for buffer in (data, data.tobytes(), bytearray(data), memoryview(data), data.view(np.float32), data[::2], data[:0], 7):
        got, want = outcome_of(pyhost.decode_weights_to_device, buffer, specs), outcome_of(general, buffer, specs)
        assert got == want, (specs, type(buffer), got, want)
check(lib.tfhip_shutdown())   # the general function's own error, or its own way back
pyhost._initialised = False
assert outcome_of(pyhost.decode_weights_to_device, data, cases[0]) == outcome_of(general, data, cases[0])
assert errors()[0] == 0, errors()
"""


def test_decode_weights_to_device_is_the_general_function():
    run(DECODE)


RACE = """
data = np.zeros(1 << 20, dtype=np.uint8)
def manifest():
    return [dict(name="t%d" % i, shape=[16, 8], dtype="float32", quantization=dict(dtype="uint8", scale=0.5, min=-1.0)) for i in range(400)]
def loaded(change):
    '''what comes back where another thread changes the manifest while the call waits for the upload'''
    specs = manifest()
    def other():
        while not fake.fake_hip_copies_now():
            time.sleep(0.0005)
        change(specs)
    thread = threading.Thread(target=other)
    thread.start()
    fake.fake_hip_copy_delay(50000)
    got = pyhost.decode_weights_to_device(data, specs)
    fake.fake_hip_copy_delay(0)
    thread.join()
    seen = [(name, buf.nbytes, shape) for name, (buf, shape) in got.items()]
    for buf, _ in got.values():
        buf.free()
    return specs, seen
"""


@pytest.mark.parametrize("change", [
    "specs.clear()", "specs.__delitem__(slice(10, None))", "[s.clear() for s in specs]", "[s['shape'].__setitem__(0, 1 << 30) for s in specs]",
    "[s['shape'].clear() for s in specs]", "[s.update(name='x') for s in specs]", "specs.__setitem__(slice(None), [None] * 400)",
])
def test_the_manifest_is_what_it_was_when_the_call_began(change):
    run(BODY + RACE + """
want = [("t%d" % i, 512, [16, 8]) for i in range(400)]
specs, got = loaded(lambda specs: """ + change + """)
assert got == want
assert specs != manifest(), "the other thread came too late"
""")


def test_a_keys_own_comparison_may_shorten_the_manifest():
    # (a key with the hash of "name": the lookup asks it, and it takes the entries away)
    run(BODY + RACE + """
class Key:
    def __hash__(self):
        return hash("name")
    def __eq__(self, other):
        if armed:
            specs.clear()
        return False
armed, specs = False, manifest()
specs[0] = dict([(Key(), 1)] + list(specs[0].items()))
armed = True
try:
    pyhost.decode_weights_to_device(data, specs)
except Exception as e:
    assert isinstance(e, (KeyError, RuntimeError, TypeError, IndexError)), e
assert not specs
""")


def test_the_shape_that_comes_back_is_the_callers_own():
    run(BODY + RACE + """
specs = manifest()
got = pyhost.decode_weights_to_device(data, specs)
got["t0"][1].append(3)
assert specs[0]["shape"] == [16, 8] and got["t1"][1] == [16, 8]
""")


@pytest.mark.parametrize("wrapped", [0, 1, 399])
def test_blocks_that_find_no_owner_are_given_back(wrapped):
    run(BODY + RACE + """
left = 2 * """ + str(wrapped) + """   # attributes that may still be set
def refuse(self, name, value):
    global left
    if left == 0:
        raise MemoryError("no room for " + name)
    left -= 1
    object.__setattr__(self, name, value)
live = pyhost.memory_info()["live"]
DeviceBuffer.__setattr__ = refuse
try:
    pyhost.decode_weights_to_device(data, manifest())
    raise AssertionError("the buffers were wrapped")
except MemoryError as e:
    assert str(e) == "no room for nbytes"
del DeviceBuffer.__setattr__
assert pyhost.memory_info()["live"] == live
assert errors()[0] == 0, errors()
""")


def test_the_package_does_without_an_extension_that_does_not_load(tmp_path):
    junk = tmp_path / os.path.basename(capi.PYCALL_PATH)
    assert capi._load_pycall(str(junk)) is None
    junk.write_bytes(b"not a library")
    with pytest.warns(RuntimeWarning, match="through ctypes"):
        assert capi._load_pycall(str(junk)) is None
    # the whole package, with such a file in the place of its own
    code = """
import sys, os
sys.path.insert(0, %r)
import importlib.util
exists, of = os.path.exists, importlib.util.spec_from_file_location
importlib.util.spec_from_file_location = lambda name, path, *more: of(name, %r if "_pycall" in path else path, *more)
from tfjs_amd import capi, pyhost
assert capi.pycall is None and pyhost.device_fused_matmul.__class__ is capi.load_library.__class__
assert capi.load_library().tfhip_free(None) != 0
""" % (ROOT, str(junk))
    done = subprocess.run([sys.executable, "-W", "ignore", "-c", code], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert done.returncode == 0, done.stdout


def test_the_build_does_without_an_extension_that_does_not_compile(tmp_path, monkeypatch, capsys):
    older = tmp_path / "_pycall.so"
    monkeypatch.setattr(build, "PYCALL", str(older))
    for include in (str(tmp_path / "none"), str(tmp_path)):   # no Python.h; one that is of no use
        older.write_bytes(b"of an older build")
        monkeypatch.setattr(sysconfig, "get_paths", lambda: dict(include=include))
        assert build.build_pycall() is None and not older.exists()
        (tmp_path / "Python.h").write_text("#error of no use\n")
    assert "through ctypes" in capsys.readouterr().out


def test_the_extension_needs_nothing_newer_than_python_3_9():
    with open(os.path.join(ROOT, "tfjs_amd", "csrc", "pycall.cc")) as f:
        text = f.read()
    for newer in ("Py_NewRef", "Py_XNewRef", "PyModule_AddObjectRef", "PyType_GetModule", "Py_Is("):
        assert newer not in text


def test_an_extension_for_other_entry_points_is_not_used(tmp_path):
    # compiled against a header in which one entry point has an argument more
    header = open(os.path.join(ROOT, "include", "tfjs_hip.h")).read()
    at = header.index("int tfhip_mean_hw(") + len("int tfhip_mean_hw(")
    (tmp_path / "tfjs_hip.h").write_text(header[:at] + "int more, " + header[at:])
    other = tmp_path / os.path.basename(capi.PYCALL_PATH)
    subprocess.check_call(["g++", "-O0", "-std=c++17", "-fPIC", "-shared", "-I", sysconfig.get_paths()["include"], "-I", str(tmp_path),
                           os.path.join(ROOT, "tfjs_amd", "csrc", "pycall.cc"), "-o", str(other)])
    with pytest.warns(RuntimeWarning, match="of another build"):
        assert capi._load_pycall(str(other)) is None
    assert {name: capi._codes(capi.SIGNATURES[name]) for name in capi.pycall.NAMES} == capi.pycall.NAMES


@pytest.mark.parametrize("name", ["device_fused_matmul", "decode_weights_to_device"])
def test_the_compiled_functions_are_functions_to_the_rest_of_python(name):
    run(BODY + """
import copy, inspect, pickle, types, weakref
f = pyhost.""" + name + """
assert type(f) is not types.FunctionType, "not the compiled one"
for protocol in range(pickle.HIGHEST_PROTOCOL + 1):
    for pickler in (pickle.dumps, pickle._dumps):
        assert pickle.loads(pickler(f, protocol)) is f
assert copy.copy(f) is f and copy.deepcopy({"f": f})["f"] is f
assert weakref.ref(f)() is f
assert repr(f).startswith("<function """ + name + """ at ")
assert inspect.isfunction(f) and f.__module__ == "tfjs_amd.pyhost" and list(inspect.signature(f).parameters)
f.note = 3
assert f.note == 3
class Holder:
    method = f
assert Holder.method is f and Holder().method.__func__ is f
""")


def test_the_ctypes_functions_are_what_they_were():
    run(BODY + """
import pickle, weakref
f, p = lib.tfhip_free, plain.tfhip_free
assert type(f) is not type(p), "not the compiled one"
assert weakref.ref(f)() is f and repr(f) == repr(f.__call__.__self__)
assert ctypes.cast(f, ctypes.c_void_p).value == ctypes.cast(p, ctypes.c_void_p).value
try:
    pickle.dumps(f)
    raise AssertionError("pickled")
except ValueError as e:
    assert "pointers" in str(e)
seen = []
lib.tfhip_mean_hw.errcheck = lambda status, fn, args: seen.append((status, args)) or 77
assert lib.tfhip_mean_hw(a.ptr, out.ptr, 1, 7, 7, 16) == 77 and seen[0][0] == 0
del lib.tfhip_mean_hw.errcheck
lib.tfhip_mean_hw.restype = ctypes.c_bool
assert lib.tfhip_mean_hw(a.ptr, out.ptr, 1, 7, 7, 16) is False
""")
