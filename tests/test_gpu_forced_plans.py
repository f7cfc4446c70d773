"""The GEMM kernels on plans of the test's choice (tile height, form, split of K), which the
automatic plan would mix: every kpair tile in every output mode, split and unsplit, at the
edges of its rows, and the 128- and 256-row tiles on a split that ends with an octet of one
group.  Every row and column against the oracle.

fp32 outputs: the 2-norm of the error within KPAIR_REL of the result's for the kpair tiles
(measured 0.3e-6 to 1.4e-6 on these shapes, 2.1e-6 at K = 15360; X_g in two bf16 parts
instead of three would by itself give 1.5e-5 to 1.9e-5 on each of them), the other GEMM
tests' bar on the largest error for the larger tiles, whose X_g has two parts.  bf16
outputs: the correctly rounded value of something within 1e-4 of the RMS; GeGLU as
test_gpu_geglu.py."""

import numpy as np
import pytest
from oracle import affine as A
from oracle import c_oracle as C
from plan_host import Forced
from test_gpu_geglu import _check, _exact_gu
from test_gpu_parity import assert_close, dev_triple, dev_x, host_bits, random_triple

pytestmark = pytest.mark.gpu

KPAIR_REL = 5e-6
GEMM_REL = 5e-4


def _triple(n, k, bits, seed):
    if bits == 4:
        return random_triple(n, k, seed)
    w = A.round_to_bf16((np.random.default_rng(seed).standard_normal((n, k)) * 0.02).astype(np.float32))
    return C.quantize(w, bits=8)


def _rel(y, want):
    return float(np.linalg.norm(y.cpu().numpy().astype(np.float64) - want) / np.linalg.norm(want))


# (n, k): a ragged last row block and pair; less than one step and one row block; several
# column tiles; K of one octet and one group; N within a tile's first wave
SHAPES = [(300, 704, 4), (40, 64, 4), (520, 3840, 4), (2064, 1024, 4), (130, 576, 4), (300, 704, 8), (272, 1984, 8)]


@pytest.mark.parametrize("kmt", [2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("n,k,bits", SHAPES)
def test_kpair_tile(gpu_lib, n, k, bits, kmt):
    bm = 16 * kmt
    tri = _triple(n, k, bits, n + k + bits)
    f = Forced([dev_triple(*tri)], n, k, bits)
    octets = (k // 64 * (bits // 4) + 7) // 8
    for m in (1, bm - 1, bm, bm + 1, 2 * bm + 5):
        x = A.make_activations(m, k, seed=m + k, outliers=True)
        want = C.qmm_f64(x, *tri, bits=bits)
        xd = dev_x(x)
        for splits in sorted({1, 2, 3, octets}):
            y32, y16 = f.gemm(xd, True, bm, True, splits), f.gemm(xd, False, bm, True, splits)
            if y32 is None:
                continue
            what = f"m={m} splits={splits}"
            assert _rel(y32, want) < KPAIR_REL, (what, _rel(y32, want))
            assert_close(y32, want, what)
            ok, worst, frac = A.check_bf16_rounding(host_bits(y16), want, 1e-4)
            assert ok, (what, worst, frac)


@pytest.mark.parametrize("kmt", [2, 3, 4, 5, 6, 7])
def test_kpair_geglu(gpu_lib, kmt):
    f_out, k, bm = 1003, 1344, 16 * kmt
    gate, up = random_triple(f_out, k, 51), random_triple(f_out, k, 52)
    f = Forced([dev_triple(*gate), dev_triple(*up)], f_out, k)
    for m in (bm - 3, bm + 1):
        x = A.make_activations(m, k, seed=53 + m, outliers=True)
        g, u = _exact_gu(x, gate, up)
        for splits in (1, 3):
            for f32 in (False, True):
                _check(f.gemm(dev_x(x), f32, bm, True, splits), g, u, f"m={m} splits={splits} f32={f32}")


@pytest.mark.parametrize("kmt", [2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("rank,slices", [(4, 1), (16, 3), (28, 8), (32, 2)])
def test_kpair_lora(gpu_lib, kmt, rank, slices):
    """The delta added in the epilogue: t summed over its slices in order, t . B^T in fp32."""
    import torch

    n, k, bm = 300, 704, 16 * kmt
    tri = random_triple(n, k, 71)
    f = Forced([dev_triple(*tri)], n, k)
    rng = np.random.default_rng(rank + kmt)
    b = (rng.standard_normal((n, rank)) * 0.05).astype(np.float32)
    for m in (bm - 3, 2 * bm + 1):
        x = A.make_activations(m, k, seed=m)
        t = rng.standard_normal((slices, m, rank)).astype(np.float32)
        lora = (torch.from_numpy(t).cuda(), torch.from_numpy(b).cuda(), 2.0)
        base = C.qmm_f64(x, *tri)
        delta = t.astype(np.float64).sum(axis=0) @ b.astype(np.float64).T * 2.0
        y32 = f.gemm(dev_x(x), True, bm, True, 1, lora=lora)
        assert _rel(y32, base + delta) < KPAIR_REL, (m, _rel(y32, base + delta))
        y16 = A.bf16_bits_to_f32(host_bits(f.gemm(dev_x(x), False, bm, True, 1, lora=lora))).astype(np.float64)
        want = A.round_to_bf16((A.round_to_bf16(base.astype(np.float32)) + A.round_to_bf16(delta.astype(np.float32))))
        want = want.astype(np.float64)
        # base and delta each rounded, then their sum: an ulp of either part and of the sum
        ulp = A.bf16_ulp(want) + A.bf16_ulp(base) + A.bf16_ulp(delta)
        assert (np.abs(y16 - want) <= ulp).all(), m
        assert np.mean(y16 == want) > 0.97, m


# 57 groups: seven whole octets and a last one of one group.  Where a split of two or more
# octets ends on it, that octet's one step also applies the previous octet's bias term, so
# the 128-row tile writes its group sums of x after the loop and the 256-row tile loads
# them there from the pre-pass; with eight splits the octet is a split of its own.
@pytest.mark.parametrize("bm,kpair,form", [(128, False, 0), (256, False, 0), (256, False, 1), (32, True, 0), (112, True, 0)])
@pytest.mark.parametrize("splits", [1, 3, 4, 8])
def test_last_octet_of_one_group(gpu_lib, bm, kpair, form, splits):
    n, k, m = 520, 57 * 64, 300
    tri = random_triple(n, k, 5700)
    top = int((np.asarray(tri[1]).astype(np.int32) >> 7 & 0xFF).max())
    f = Forced([dev_triple(*tri)], n, k)
    x = A.make_activations(m, k, seed=5800, outliers=True)
    want = C.qmm_f64(x, *tri)
    p = 12 - (top - 127) if form == 1 else 0
    y32, y16 = (f.gemm(dev_x(x), f32, bm, kpair, splits, form, p) for f32 in (True, False))
    assert y32 is not None
    assert assert_close(y32, want, f"{bm} rows, {splits} splits") < GEMM_REL
    assert_close(y16, want, f"{bm} rows, {splits} splits")
    if kpair:
        assert _rel(y32, want) < KPAIR_REL, _rel(y32, want)


# two octets of a plane each ending raggedly, in one pass over both planes of 8-bit handles
@pytest.mark.parametrize("bm", [128, 256])
@pytest.mark.parametrize("k,splits", [(18 * 64, 1), (18 * 64, 3), (26 * 64, 2)])
def test_one_pass_ragged_octets(gpu_lib, bm, k, splits):
    n, m = 300, 270
    tri = _triple(n, k, 8, k)
    f = Forced([dev_triple(*tri)], n, k, 8)
    x = A.make_activations(m, k, seed=k, outliers=True)
    want = C.qmm_f64(x, *tri, bits=8)
    y32 = f.gemm(dev_x(x), True, bm, False, splits, 2)
    assert assert_close(y32, want, f"{bm} rows, {splits} splits") < GEMM_REL
