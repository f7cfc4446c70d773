"""The greedy head's reduction over its 16-row blocks' keys at the edges of a round of
16384 keys (1024 threads of 16): fewer keys than threads, the last key alone in its round,
and more than one round.  Token and value are exactly the first maximum of the logits that
the same call returns."""

import numpy as np
import pytest
from test_gpu_parity import dev_x
from oracle import affine as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [16, 40, 16 * 1024 + 3, 262144 - 16, 262144 + 5, 262144 + 16 * 1500])
def test_greedy_reduce_rounds(gpu_lib, n):
    import torch

    k, m = 64, 3
    g = torch.Generator(device="cuda").manual_seed(n)
    w = torch.randint(-2 ** 31, 2 ** 31 - 1, (n, k // 8), dtype=torch.int32, device="cuda", generator=g)
    s = (torch.rand((n, 1), device="cuda", generator=g) * 0.01 + 0.002).bfloat16()
    b = (-7.5 * s.float()).bfloat16()
    lin = gpu_lib.QuantizedLinear(w, s, b)
    x = dev_x(A.make_activations(m, k, seed=7))
    for where in (0, n // 2, n - 1):  # a clear maximum in the first, a middle and the last block
        s2, b2 = s.clone(), b.clone()
        b2[where] = 8.0
        x2 = x.abs()
        big = gpu_lib.QuantizedLinear(w, s2, b2)
        token, value, logits = big.forward_greedy(x2, return_logits=True)
        torch.cuda.synchronize()
        assert (token == where).all(), (n, where, token)
        assert torch.equal(value, logits.float().amax(dim=1))
        big.close()
    token, value, logits = lin.forward_greedy(x, softcap=0.0, return_logits=True)
    torch.cuda.synchronize()
    lg = logits.float().cpu().numpy()
    assert (token.cpu().numpy() == lg.argmax(axis=1)).all()
    assert np.array_equal(value.cpu().numpy(), lg.max(axis=1))
    lin.close()
