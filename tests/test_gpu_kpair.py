"""GPU parity of calls that take the kpair GEMM (q4_gemm_kpair.hip) with the plan they get
(at these small shapes mostly its 32-row tile; test_gpu_forced_plans.py runs every tile and
split), against the oracle on every row and against the decode path of the same handle (the
general path of those sizes).  fp32 outputs: the 2-norm of the error within KPAIR_REL of the
result's (fp32 sums, X_g in three bf16 parts), and within 2 ACC_REL of the RMS of the decode
path's; bf16 and GeGLU with the other GEMM tests' bars."""

import numpy as np
import pytest
from oracle import affine as A
from oracle import c_oracle as C
from test_gpu_forced_plans import KPAIR_REL, _rel
from test_gpu_parity import ACC_REL, assert_close, dev_triple, dev_x, random_triple

pytestmark = pytest.mark.gpu

# (n, k): a ragged last row block and group pair; fewer groups than a step; a split of K;
# many row blocks; K of one octet and one group
SHAPES = [(300, 704), (40, 64), (520, 3840), (2064, 1024), (130, 576)]


@pytest.fixture
def from_one(gpu_lib):
    prev = gpu_lib.set_gemm_min_rows(1)
    yield gpu_lib
    gpu_lib.set_gemm_min_rows(prev)


@pytest.mark.parametrize("n,k", SHAPES)
@pytest.mark.parametrize("bits", [4, 8])
def test_kpair_rows(from_one, n, k, bits):
    import torch

    rng = np.random.default_rng(n + k + bits)
    w = A.round_to_bf16((rng.standard_normal((n, k)) * 0.02).astype(np.float32))
    tri = C.quantize(w, bits=bits)
    lin = from_one.QuantizedLinear(*dev_triple(*tri), bits=bits)
    for m in (1, 15, 17, 32, 33, 48, 49, 80, 81, 111, 112, 113, 225):
        x = A.make_activations(m, k, seed=m + k, outliers=True)
        want = C.qmm_f64(x, *tri, bits=bits)
        xd = dev_x(x)
        y32, y16 = lin.forward(xd, out_dtype=torch.float32), lin.forward(xd)
        guard = torch.full((m + 3, n), -7.0, device="cuda")
        lin.forward(xd, out=guard[:m])
        from_one.set_gemm_min_rows(1 << 20)
        dec = lin.forward(xd, out_dtype=torch.float32)
        from_one.set_gemm_min_rows(1)
        torch.cuda.synchronize()
        assert assert_close(y32, want, f"m={m} fp32") < ACC_REL
        assert _rel(y32, want) < KPAIR_REL, f"m={m}: {_rel(y32, want)}"
        assert_close(y16, want, f"m={m} bf16")
        rms = float(np.sqrt(np.mean(want ** 2)))
        assert float((y32 - dec).abs().max()) <= 2 * ACC_REL * rms, f"m={m}: differs from the decode path"
        assert torch.equal(guard[:m], y32) and bool((guard[m:] == -7.0).all()), f"m={m}: rows past M written"
    lin.close()


@pytest.mark.parametrize("m", [17, 45, 112, 200, 300])
def test_kpair_pair(from_one, m):
    """GeGLU of a pair, both dtypes (unsplit plans; after a split: test_gpu_forced_plans.py)."""
    import torch

    from test_gpu_geglu import _check, _exact_gu

    f, k = 1003, 1344
    gate, up = random_triple(f, k, 51), random_triple(f, k, 52)
    pair = from_one.QuantizedGeGLU(dev_triple(*gate), dev_triple(*up))
    x = A.make_activations(m, k, seed=53 + m, outliers=True)
    h16, h32 = pair.forward(dev_x(x)), pair.forward(dev_x(x), out_dtype=torch.float32)
    torch.cuda.synchronize()
    rows = np.arange(m)
    g_exact, u_exact = _exact_gu(x, gate, up, rows)
    _check(h16, g_exact, u_exact, f"m={m}")
    _check(h32, g_exact, u_exact, f"m={m} fp32")
    pair.close()


def test_kpair_special_values(from_one):
    """Rows with inf, NaN, subnormals and the largest values do not touch other rows."""
    import torch

    n, k, m = 272, 640, 50
    tri = random_triple(n, k, 61)
    lin = from_one.QuantizedLinear(*dev_triple(*tri))
    x = A.make_activations(m, k, seed=62)
    clean = lin.forward(dev_x(x), out_dtype=torch.float32)
    x2 = x.copy()
    x2[3, 5], x2[17, 600], x2[40, :] = 0x7F80, 0x7FC0, 0x0001
    y = lin.forward(dev_x(x2), out_dtype=torch.float32)
    torch.cuda.synchronize()
    keep = np.setdiff1d(np.arange(m), [3, 17, 40])
    kt = torch.from_numpy(keep).cuda()
    assert torch.equal(y[kt], clean[kt])
    assert not bool(torch.isfinite(y[3]).any()) and bool(torch.isnan(y[17]).all())
    want = C.qmm_f64(x2[40:41], *tri)
    assert np.abs(y[40].cpu().numpy() - want[0]).max() <= 1e-37
    lin.close()
