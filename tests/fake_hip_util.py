"""Runs Python code against libtfjs_hip.so with a stand-in for the HIP runtime (tests/fake_hip/fake_hip.cc): the
library's host code without a GPU. Every snippet gets a process of its own, in which the stand-in is loaded into the
global scope first, so that the library's calls reach it and not the runtime it was linked with."""
import os
import subprocess
import sys
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = os.path.join(ROOT, "tests", "fake_hip", "fake_hip.cc")

PRELUDE = """
import ctypes, os, sys, threading, time
sys.path.insert(0, %r)
fake = ctypes.CDLL(%r, mode=ctypes.RTLD_GLOBAL)
import numpy as np
from tfjs_amd import capi, pyhost
from tfjs_amd.capi import DeviceBuffer, check, i64_array
lib = capi.load_library()

def launch(back=0):
    '''(kernel, device, recorded, leading words of the first argument) of an earlier launch'''
    name, words, recorded = ctypes.create_string_buffer(512), (ctypes.c_uint64 * 24)(), ctypes.c_int()
    device = fake.fake_hip_launch(back, name, 512, words, ctypes.sizeof(words), ctypes.byref(recorded))
    return name.value.decode(), device, bool(recorded.value), list(words)

def errors():
    text = ctypes.create_string_buffer(512)
    return fake.fake_hip_errors(text, 512), text.value.decode()
"""

_built = None


def _stand_in():
    global _built
    if _built is None:
        folder = tempfile.TemporaryDirectory(prefix="fake_hip_")
        out = os.path.join(folder.name, "libfake_hip.so")
        subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__",
                               "-I/opt/rocm/include", SOURCE, "-o", out])
        _built = (folder, out)
    return _built[1]


def run(body, each=([],), timeout=60):
    """Runs `body` behind PRELUDE, once for each list of arguments; fails where it fails or does not end."""
    code = PRELUDE % (ROOT, _stand_in()) + body
    for args in each:
        done = subprocess.run([sys.executable, "-c", code] + args, stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                              text=True, timeout=timeout)
        assert done.returncode == 0, done.stdout[-4000:]
