"""ctypes access to the library's path choice and GEMM plan (no GPU needed: without one the
plan takes 256 compute units), and GEMM launches with a plan of the test's choice."""

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
                            "-I", hbuild.CSRC, deps[0], "-L", hbuild.LIB_DIR, "-l:" + hbuild.LIB_NAME,
                            "-Wl,-rpath,$ORIGIN/../../helios_amd/lib", "-o", SO], check=True, capture_output=True)
        _fn = ctypes.CDLL(SO)
        i, p, ul = ctypes.c_int, ctypes.c_void_p, ctypes.c_ulong
        _fn.q4_route.argtypes = [i] * 7 + [ul, ctypes.POINTER(ctypes.c_long)]
        _fn.q4_rec_bytes.argtypes, _fn.q4_rec_bytes.restype = [i] * 4, ul
        _fn.q4_repack.argtypes = [p] * 4 + [i] * 4 + [p]
        _fn.q4_gelu.argtypes = [p, p]
        _fn.q4_forced_bytes.argtypes, _fn.q4_forced_bytes.restype = [i] * 9, ctypes.c_long
        _fn.q4_forced_gemm.argtypes = [p, p, p] + [i] * 11 + [p, ul, p, p, p, i, i, ctypes.c_float, p]
    return _fn


def route(n, k, rows, bits=4, pair=False, f16=True, min_rows=0, room=2 ** 64 - 1) -> dict:
    """What a forward of `rows` rows runs on (N or, for a pair, F; K).  f16: the handle's
    scales allow the fp16 form."""
    out = (ctypes.c_long * 7)()
    _load().q4_route(n, k, bits, int(pair), int(f16), rows, min_rows, room, out)
    return dict(zip(NAMES, out))


class Forced:
    """One projection (or gate|up pair) repacked as the library's handles are, and GEMM
    launches on it with a given tile, form and split of K.  Outputs lie in a buffer with
    guards on both sides, which every launch must leave alone."""

    GUARD = 512

    def __init__(self, triples, n, k, bits=4):
        import torch

        self.lib, self.n, self.k, self.bits, self.pair = _load(), n, k, bits, len(triples) == 2
        self.stream = torch.cuda.current_stream().cuda_stream
        self.tiles = torch.empty(self.lib.q4_rec_bytes(n, k, bits, self.pair), dtype=torch.uint8, device="cuda")
        ptrs = [(ctypes.c_void_p * 2)(*[t[j].data_ptr() for t in triples]) for j in range(3)]
        assert self.lib.q4_repack(*ptrs, self.tiles.data_ptr(), n, k, bits, self.pair, self.stream) == 0
        self.gelu = torch.empty(2 * 11 * 128, dtype=torch.int16, device="cuda")
        assert self.lib.q4_gelu(self.gelu.data_ptr(), self.stream) == 0
        torch.cuda.synchronize()

    def gemm(self, x, f32, bm, kpair, splits, form=0, f16_p=0, lora=None):
        """y (h for a pair) of x [m, k], or None where K has no such split.  lora: (t
        [slices, m, rank] fp32, B [n, rank] fp32, scale)."""
        import torch

        m = x.shape[0]
        args = (self.n, self.k, self.bits, int(self.pair))
        need = self.lib.q4_forced_bytes(*args, m, bm, int(kpair), form, splits)
        if need < 0:
            return None
        assert x.shape == (m, self.k) and x.is_contiguous() and x.dtype == torch.bfloat16
        dtype = torch.float32 if f32 else torch.bfloat16
        # guards before and after, and an output aligned to its elements only
        buf = torch.full((m * self.n + 2 * self.GUARD + 1,), -7.0, dtype=dtype, device="cuda")
        y = buf[self.GUARD + 1:self.GUARD + 1 + m * self.n]
        y.fill_(float("nan"))
        ws = torch.full((need // 4 + 64,), float("nan"), device="cuda")
        t, b, scale = lora if lora is not None else (None, None, 0.0)
        mode = int(f32) + (2 if self.pair else 0)
        rc = self.lib.q4_forced_gemm(self.tiles.data_ptr(), x.data_ptr(), y.data_ptr(), m, mode, *args, f16_p, bm, int(kpair), form,
                                     splits, ws.data_ptr(), need, self.gelu.data_ptr(), t.data_ptr() if t is not None else None,
                                     b.data_ptr() if b is not None else None, t.shape[2] if t is not None else 0,
                                     t.shape[0] if t is not None else 0, scale, self.stream)
        assert rc == 0, rc
        torch.cuda.synchronize()
        assert bool((buf[:self.GUARD + 1] == -7.0).all()) and bool((buf[self.GUARD + 1 + m * self.n:] == -7.0).all()), \
            "written outside the output"
        assert bool((ws[need // 4:] != ws[need // 4:]).all()), "written past the scratch"
        return y.view(m, self.n)
