"""Runs a test's body in a child process in which the library's HIP calls go to
a host model of the runtime (hip_model.cpp): for host code whose faults a GPU
must not be driven into, or that needs a second device."""
import ctypes
import functools
import os
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

FAIL_LAUNCH, HOST_BYTES, DELAY_FLAG = range(3)  # model_set's keys
PORTABLE, COHERENT, NONCOHERENT = 0x1, 0x40000000, 0x80000000  # hipHostMalloc's flags
REGISTER_READ_ONLY = 0x8  # of hipHostRegister's


@functools.lru_cache(maxsize=1)
def _library():
    out = os.path.join(tempfile.mkdtemp(prefix="hip_model_"), "libhip_model.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-w", "-pthread", "-I/opt/rocm/include",
                    os.path.join(HERE, "hip_model.cpp"), "-o", out], check=True)
    return out


def modelled(body):
    """the test runs body(model, rt) in a child process"""

    @functools.wraps(body)
    def test():
        r = subprocess.run([sys.executable, "-c", _CHILD, _library(), body.__module__, body.__name__],
                           capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]

    del test.__wrapped__  # pytest looks for fixtures in the body's arguments
    test.body = body
    return test


_CHILD = f"""
import ctypes, importlib, sys
sys.path[:0] = [{HERE!r}, {ROOT!r}]
m = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
m.model_launched.restype = ctypes.c_char_p
m.model_common_flags.restype = ctypes.c_uint
m.model_host_bytes.restype = m.model_host_blocks.restype = m.model_host_allocs.restype = ctypes.c_long
m.model_set.argtypes = [ctypes.c_int, ctypes.c_long]
m.model_lock.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_uint]
m.launched = lambda: m.model_launched().decode().split()
from emma_amd import rt
rt.load()
assert rt.device_count() == 2, "the library's HIP calls do not reach the model"
getattr(importlib.import_module(sys.argv[2]), sys.argv[3]).body(m, rt)
"""
