"""Runs programs through the native library's host side on the CPU: its sources linked against a
HIP runtime without a device (hip_stub.cpp).  Kernels are emitted and built for gfx950 by hiprtc as
always; launches are recorded instead of run, so tensors may be views of any size over a small
buffer."""

import contextlib
import ctypes
import hashlib
import os
import subprocess
import time
from dataclasses import dataclass

import pto_wsp._hip as _hip
from pto_wsp import _build

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(HERE, "_build", "libptowsp_stub.so")


def _library():
    srcs = [os.path.join(_build.CSRC, "host", s) for s in _build.HOST_SOURCES if s.endswith(".cpp")]
    srcs.append(os.path.join(HERE, "hip_stub.cpp"))
    _build._write_embedded_headers()
    host = os.path.join(_build.CSRC, "host")
    read = srcs + [os.path.join(host, f) for f in sorted(os.listdir(host)) if f.endswith(".hpp")]
    read += [os.path.join(_build.BUILD_DIR, "device_headers.inc"), os.path.join(_build.INCLUDE, "ptowsp_hip.h"),
             os.path.join(_build.INCLUDE, "ptowsp_abi.h")]
    key = hashlib.sha256(b"".join(open(p, "rb").read() for p in read)).hexdigest()[:16]
    path = LIB.replace(".so", f"_{key}.so")
    if not os.path.exists(path):
        os.makedirs(os.path.dirname(path), exist_ok=True)
        for old in os.listdir(os.path.dirname(path)):
            if old.startswith("libptowsp_stub") and old.endswith(".so"):
                os.unlink(os.path.join(os.path.dirname(path), old))
        procs = []
        for s in srcs:
            o = f"{path}.{os.getpid()}.{os.path.basename(s)}.o"
            cmd = ["hipcc", "--offload-host-only", "-O2", "-std=c++17", "-fPIC", "-w", "-I", _build.INCLUDE, "-I", _build.BUILD_DIR, "-I", host,
                   "-c", s, "-o", o]
            procs.append((subprocess.Popen(cmd), o))
        assert all(p.wait() == 0 for p, _ in procs)
        objs = [o for _, o in procs]
        subprocess.run(["g++", "-shared", "-Wl,-Bsymbolic", *objs, "-o", f"{path}.{os.getpid()}.tmp", "-L/opt/rocm/lib", "-lhiprtc",
                        "-Wl,-rpath,/opt/rocm/lib"], check=True)
        for o in objs:
            os.unlink(o)
        os.replace(f"{path}.{os.getpid()}.tmp", path)
    lib = ctypes.CDLL(path)
    for name, f in vars(_hip._lib).items():
        if name.startswith("ptowsp_"):
            getattr(lib, name).argtypes, getattr(lib, name).restype = f.argtypes, f.restype
    lib.stub_entry.restype = ctypes.c_char_p
    for name in ("stub_blocks", "stub_threads"):
        getattr(lib, name).restype = ctypes.c_uint64
    lib.stub_base.restype = ctypes.c_void_p
    lib.stub_freed.argtypes = [ctypes.c_void_p]
    for name in ("stub_s3", "stub_s4", "stub_coef"):
        getattr(lib, name).restype = ctypes.c_int64
    return lib


_lib = None


@dataclass
class Launch:
    entry: str
    blocks: int
    threads: int
    s3: list
    s4: list
    coef: list
    base: list


def recorded():
    """Entry points of the launches of the last pass, also of one that failed."""
    return [_lib.stub_entry(i).decode() for i in range(_lib.stub_num_launches())]


def _launches(prog):
    out = []
    for i in range(_lib.stub_num_launches()):
        out.append(Launch(_lib.stub_entry(i).decode(), _lib.stub_blocks(i), _lib.stub_threads(i),
                          [_lib.stub_s3(i, p) for p in range(12)], [_lib.stub_s4(i, p) for p in range(12)],
                          [[_lib.stub_coef(i, p, v) for v in range(8)] for p in range(12)], [_lib.stub_base(i, p) for p in range(12)]))
    assert prog.stats.launches == len(out)
    return out


def freed(pointer):
    """Whether device memory that a launch was given has been freed."""
    return bool(_lib.stub_freed(pointer))


@contextlib.contextmanager
def program(workload):
    """`workload` compiled for the recorded runtime: a function that runs it once (capture: on a stream
    that is being captured) and returns its launches."""
    global _lib
    if _lib is None:
        _lib = _library()
    real, _hip._lib = _hip._lib, _lib
    prog = None

    def once(capture=False):
        _lib.stub_clear()
        _lib.stub_capture(int(capture))
        try:
            prog.execute()
        finally:
            _lib.stub_capture(0)
        prog.synchronize()
        return _launches(prog)

    try:
        prog = workload.compile(target="hip_gfx950")
        once.prog = prog
        yield once
    finally:
        if prog is not None:
            prog._native.__del__()  # here and now: an exception's traceback may hold it beyond this library
        _hip._lib = real


def run(workload, passes=1):
    """Launches of one pass of `workload`, and the host time in seconds of the fastest pass after the first."""
    with program(workload) as once:
        best = 1e9
        for i in range(passes):
            t = time.perf_counter()
            launches = once()
            if i > 0 or passes == 1:
                best = min(best, time.perf_counter() - t)
        return launches, best
