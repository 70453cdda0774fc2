"""Runs a piece of Python in a process of its own whose HIP runtime is tests/cpp/host_hip.cpp: host memory, launches
logged and not executed.  No GPU is used, present or not."""
import atexit
import functools
import os
import shutil
import subprocess
import sys
import tempfile
import textwrap

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

_PRELUDE = '''
import ctypes, importlib, sys
hip = ctypes.CDLL(%(lib)r, mode=ctypes.RTLD_GLOBAL)  # in front of every library loaded later
hip.host_hip_calls.restype = ctypes.c_long
hip.host_hip_launch.restype = ctypes.c_char_p
sys.path[:0] = [%(root)r, %(here)r, %(root)r + "/oracle"]
import numpy as np
m = importlib.import_module("esp-dl_amd")
m.capi.torch_device_first = lambda: None
zoo, model = m.zoo, m.model

def launches():
    """The launches since the last host_hip_clear: kernel, grid, block, dynamic LDS bytes, LDS limit, thread."""
    out = []
    for i in range(hip.host_hip_launches()):
        sizes, thread = (ctypes.c_uint * 8)(), ctypes.c_ulonglong()
        name = hip.host_hip_launch(i, sizes, ctypes.byref(thread)).decode()
        out.append(dict(name=name, grid=tuple(sizes[0:3]), block=tuple(sizes[3:6]), lds=sizes[6], limit=sizes[7], thread=thread.value))
    return out
'''


@functools.lru_cache(maxsize=None)
def _library():
    folder = tempfile.mkdtemp(prefix="host_hip")
    atexit.register(shutil.rmtree, folder, ignore_errors=True)
    lib = os.path.join(folder, "libhost_hip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "cpp", "host_hip.cpp"), "-o", lib, "-lpthread"], check=True)
    return lib


def run(script, timeout=120):
    """Output of the script; fails when the script does."""
    text = _PRELUDE % {"lib": _library(), "root": ROOT, "here": HERE} + textwrap.dedent(script)
    r = subprocess.run([sys.executable, "-c", text], capture_output=True, text=True, timeout=timeout)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout
