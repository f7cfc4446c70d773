"""8-bit handles at the row counts where their path changes: 3 and 4 rows on wide outputs
(the int8 kernels from 512 row blocks, the bf16 ones below) and 8 to 17 rows around the
GEMM's first (9 rows from N x 2K = 1e8, 12 from 6e7).  Every automatic result against the oracle and
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
