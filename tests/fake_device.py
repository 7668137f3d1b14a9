"""The host library on tests/native/fake_hip.cpp, a HIP runtime without a device:
run(code) executes code in a process of its own, where `lib` is the library,
`fake` the runtime's test side and the functions of PRELUDE are defined.  Device
pointers are plain numbers."""
import os
import subprocess
import sys
import tempfile

import caps_amd

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "tests", "native", "fake_hip.cpp")

PRELUDE = """
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_count.restype = ctypes.c_longlong
fake.fake_free.restype = ctypes.c_size_t
fake.fake_set_free.argtypes = fake.fake_set_malloc_limit.argtypes = [ctypes.c_size_t]
import caps_amd
lib = caps_amd.load()
FP64, LEAF, CRT, BF16 = (caps_amd.MODE_FP64, caps_amd.MODE_OZAKI_INT8, caps_amd.MODE_CRT_INT8,
                         caps_amd.MODE_CRT_BF16)
GiB, MiB = 1 << 30, 1 << 20
def count(what):
    return fake.fake_count(what.encode())
def opts(mode, moduli=0, flags=0, cutoff=0):
    return caps_amd.Options(mode, moduli, flags, cutoff)
def call(n, r, pattern, mode=FP64, bs=1, moduli=0, flags=0, at=1, entry=None, cutoff=0,
         stream=None):
    d, o = caps_amd.MatDescriptor.one_device(n, r, bs), opts(mode, moduli, flags, cutoff)
    p = [(at << 44) + (k << 40) for k in range(3)]
    f = entry or lib.caps_multiply_device
    return f(*p, ctypes.byref(d), pattern.encode() if pattern else None, ctypes.byref(o), stream)
def batch(shapes, mode=FP64, at=1, stream=None):
    k = len(shapes)
    ptr = [(ctypes.c_void_p * k)(*[(at << 44) + (s << 41) + (i << 32) for i in range(k)])
           for s in range(3)]
    descs = (caps_amd.MatDescriptor * k)(*[caps_amd.MatDescriptor.one_device(n, r)
                                           for n, r, _ in shapes])
    pats = (ctypes.c_char_p * k)(*[p.encode() if p else None for _, _, p in shapes])
    os_ = (caps_amd.Options * k)(*[opts(mode) for _ in shapes])
    return lib.caps_multiply_batch_device(k, *[ctypes.cast(x, ctypes.c_void_p) for x in ptr],
                                          ctypes.cast(descs, ctypes.c_void_p),
                                          ctypes.cast(pats, ctypes.c_void_p),
                                          ctypes.cast(os_, ctypes.c_void_p), stream)
def error():
    return lib.caps_last_error().decode()
def peak_bytes():
    return caps_amd.counters()["peak_workspace_mb"] * MiB
def reported():
    return caps_amd.counters()["pattern"]
"""


def library() -> str:
    """The fake runtime, built once per version of its source."""
    path = os.path.join(tempfile.gettempdir(),
                        f"libfakehip_{os.getuid()}_{os.stat(SRC).st_mtime_ns}.so")
    if not os.path.exists(path):
        tmp = f"{path}.{os.getpid()}"
        subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                        "-I/opt/rocm/include", SRC, "-o", tmp], check=True)
        os.replace(tmp, path)
    return path


def run(code: str) -> None:
    if not os.path.exists(caps_amd.LIB_PATH):
        from caps_amd import build
        build.build()
    r = subprocess.run([sys.executable, "-c", PRELUDE + code, library()], cwd=ROOT,
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
