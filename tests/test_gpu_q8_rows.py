"""8-bit handles at the row counts where their path changes: 2 to 5 rows (the int8 kernels
up to 2, the bf16 ones from 3) and 8 to 17 rows around the
first row counts at which wide outputs go to the GEMM (9 and 12).  Every automatic result against the oracle and
against both pinned paths: fp32 outputs within GEMM_REL of the RMS (the kernels' sums are
exact products in fp32, in different orders)."""

import numpy as np
import pytest
from oracle import affine as A
from oracle import c_oracle as C
from test_gpu_parity import assert_close, dev_triple, dev_x

pytestmark = pytest.mark.gpu

GEMM_REL = 5e-4


@pytest.mark.parametrize("n,k,rows", [(8192, 256, (2, 3, 4, 5)), (8176, 320, (3, 4)), (8200, 192, (3, 4)),
                                      (8192, 3712, (9, 11, 12, 17)), (3840, 7808, (11, 12)), (3840, 7872, (12, 16)),
                                      (8192, 6144, (8, 9, 16))])
def test_q8_row_rules(gpu_lib, n, k, rows):
    import torch

    rng = np.random.default_rng(n + k)
    w = A.round_to_bf16((rng.standard_normal((n, k)) * 0.02).astype(np.float32))
    tri = C.quantize(w, bits=8)
    lin = gpu_lib.QuantizedLinear(*dev_triple(*tri), bits=8)
    for m in rows:
        x = A.make_activations(m, k, seed=m, outliers=True)
        want = C.qmm_f64(x, *tri, bits=8)
        xd = dev_x(x)
        y32, y16 = lin.forward(xd, out_dtype=torch.float32), lin.forward(xd)
        with gpu_lib.gemm_min_rows(1):
            gm = lin.forward(xd, out_dtype=torch.float32)
        with gpu_lib.gemm_min_rows(1 << 20), gpu_lib.decode_kernel(2):
            dc = lin.forward(xd, out_dtype=torch.float32)
        torch.cuda.synchronize()
        assert assert_close(y32, want, f"m={m} fp32") < GEMM_REL
        assert_close(y16, want, f"m={m} bf16")
        rms = float(np.sqrt(np.mean(want ** 2)))
        for other in (gm, dc):
            assert float((y32 - other).abs().max()) <= GEMM_REL * rms, m
    lin.close()


@pytest.mark.parametrize("n", [8192, 65536 + 16])
@pytest.mark.parametrize("m", [3, 4])
def test_q8_small_x_beside_large(gpu_lib, n, m):
    """x is taken as it is at 3-4 rows of an 8-bit handle, whatever else its group holds:
    rows of one value 1 and 63 of 0.75 x 2^-21 a group (below what 20 bits under the
    group's largest keep), and rows of bf16 subnormals only.  The large value's weight is
    exactly 0, so the result is the small values'.  fp32 sums of the factored form
    (weights as 16 s (1 + q/16) on two planes): each group's terms total at most 512 s
    sum |x|, and eight roundings of 2^-24 of that bound the error."""
    import torch

    k = 256
    rng = np.random.default_rng(n + m)
    codes = rng.integers(192, 256, (n, k)).astype(np.uint8)
    codes[:, ::64] = 128
    w = np.ascontiguousarray(codes).view(np.uint32)
    sf = A.round_to_bf16((rng.random((n, k // 64)) * 0.01 + 0.002).astype(np.float32))
    tri = (w, A.f32_to_bf16_bits(sf), A.f32_to_bf16_bits(-128.0 * sf))
    xf = np.full((m, k), 0.75 * 2.0 ** -21, np.float32)
    xf[:, ::64] = 1.0
    x = A.f32_to_bf16_bits(xf)
    x[m - 1] = rng.integers(0x20, 0x80, k)  # subnormals only
    lin = gpu_lib.QuantizedLinear(*dev_triple(*tri), bits=8)
    y = lin.forward(dev_x(x), out_dtype=torch.float32).cpu().numpy().astype(np.float64)
    lin.close()
    want = C.qmm_f64(x, *tri, bits=8)
    xs = np.abs(A.bf16_bits_to_f32(x).astype(np.float64)).reshape(m, k // 64, 64).sum(axis=2)
    bound = 8 * 2.0 ** -24 * 512 * xs @ sf.astype(np.float64).T
    assert (want > 4 * bound).all()
    worst = (np.abs(y - want) / bound).max(axis=1)
    assert (worst <= 1).all(), worst
