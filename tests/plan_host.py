"""ctypes access to the library's path choice and GEMM plan (no GPU needed: without one the
plan takes 256 compute units)."""

import ctypes
import os
import subprocess

from helios_amd import build as hbuild
from helios_amd import qmm

HERE = os.path.dirname(os.path.abspath(__file__))
SO = os.path.join(HERE, "_build", "libplanhost.so")
NAMES = ("decode", "bm", "splits", "kpair", "f16", "q8", "scratch")
_fn = None


def _load():
    global _fn
    if _fn is None:
        if not os.path.exists(hbuild.LIB_PATH):
            hbuild.build()
        qmm.load_library()
        deps = [os.path.join(HERE, "plan_host.cpp"), os.path.join(hbuild.CSRC, "q4_kernels.h"), hbuild.LIB_PATH]
        if not os.path.exists(SO) or any(os.path.getmtime(d) > os.path.getmtime(SO) for d in deps):
            os.makedirs(os.path.dirname(SO), exist_ok=True)
            subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                            "-I", hbuild.CSRC, deps[0], hbuild.LIB_PATH, "-o", SO], check=True, capture_output=True)
        _fn = ctypes.CDLL(SO).q4_route
        _fn.argtypes = [ctypes.c_int] * 7 + [ctypes.c_ulong, ctypes.POINTER(ctypes.c_long)]
    return _fn


def route(n, k, rows, bits=4, pair=False, f16=True, min_rows=0, room=2 ** 64 - 1) -> dict:
    """What a forward of `rows` rows runs on (N or, for a pair, F; K).  f16: the handle's
    scales allow the fp16 form."""
    out = (ctypes.c_long * 7)()
    _load()(n, k, bits, int(pair), int(f16), rows, min_rows, room, out)
    return dict(zip(NAMES, out))
