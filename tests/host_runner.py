"""Build libsfx's host code (argument checks, scratch, host copies) against a HIP
runtime in host memory (tests/host/fake_hip.cpp); tests only, no GPU.

Needs hipcc for the HIP headers' host pass; no device code is compiled and
the real HIP runtime is not linked.
"""
from __future__ import annotations

import ctypes as C
import os
import shutil
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "sfemans_amd", "csrc")
OUT = os.path.join(HERE, "host", "_build")
LIB = os.path.join(OUT, "libsfx_host.so")
SRCS = [os.path.join(HERE, "host", "fake_hip.cpp")] + [
    os.path.join(CSRC, f) for f in ("sfx_api.cpp", "sfx_exact_host.cpp", "sfx_hostcopy.cpp")]


def hipcc() -> str | None:
    return shutil.which("hipcc") or ("/opt/rocm/bin/hipcc" if os.path.exists("/opt/rocm/bin/hipcc") else None)


def load() -> C.CDLL:
    """The library, freshly loaded state included: one copy per call."""
    deps = SRCS + [os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".h")]
    if not (os.path.exists(LIB) and os.path.getmtime(LIB) >= max(os.path.getmtime(d) for d in deps)):
        os.makedirs(OUT, exist_ok=True)
        tag = f".tmp{os.getpid()}"
        objs = []
        for s in SRCS:
            o = os.path.join(OUT, os.path.basename(s) + tag + ".o")
            subprocess.run([hipcc(), "-x", "hip", "--offload-host-only", "-std=c++17", "-O1", "-g", "-fPIC",
                            "-I", CSRC, "-c", s, "-o", o], check=True)
            objs.append(o)
        subprocess.run(["g++", "-shared", "-pthread", "-Wl,-Bsymbolic", "-o", LIB + tag] + objs, check=True)
        os.replace(LIB + tag, LIB)
        for o in objs:
            os.remove(o)
    copy = LIB + f".{os.getpid()}.{load.n}.so"
    load.n += 1
    shutil.copyfile(LIB, copy)
    try:
        L = C.CDLL(copy, mode=os.RTLD_LOCAL | os.RTLD_NOW)
    finally:
        os.remove(copy)
    vp, i64, i32, d, z = C.c_void_p, C.c_int64, C.c_int32, C.c_double, C.c_size_t
    L.fake_count.argtypes, L.fake_count.restype = [C.c_char_p], C.c_long
    L.fake_limit.argtypes, L.fake_limit.restype = [z], None
    L.fake_used.restype = z
    L.fake_capture.argtypes, L.fake_capture.restype = [vp, i32], None
    L.fake_pin.argtypes, L.fake_pin.restype = [vp, i32], None
    L.fake_pending.restype = C.c_long
    L.host_copy_out.argtypes = [vp, vp, z]
    L.host_copy_out_meanwhile.argtypes, L.host_copy_out_meanwhile.restype = [vp, vp, z], None
    L.sfx_last_error.restype = C.c_char_p
    L.sfx_stream_release.argtypes = [vp]
    L.sfx_fft_scalar_vect_dcl_dev.argtypes = [vp, vp, vp, i64, i32, i32, i32, vp]
    L.sfx_fft_par_div_dcl_dev.argtypes = [vp, vp, vp, i64, i32, i32, vp]
    return L


load.n = 0
