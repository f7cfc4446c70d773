"""Calls that take no scratch (up to 31 rows; past that small slabs): captured on a stream the
library has not seen they are kernel nodes only, and two graphs captured on one stream may be
replayed at the same time on two others.  Every replay equals the eager call bit for bit, and
so does the allocation-free entry point."""

import numpy as np
import pytest
from oracle import affine as A
from oracle import c_oracle as C
from test_gpu_parity import dev_triple, dev_x, random_triple

import hip_graph_nodes as G

pytestmark = pytest.mark.gpu


def _triple(n, k, bits, seed):
    if bits == 4:
        return random_triple(n, k, seed)
    rng = np.random.default_rng(seed)
    return C.quantize(A.round_to_bf16((rng.standard_normal((n, k)) * 0.02).astype(np.float32)), bits=8)


@pytest.mark.parametrize("n,k,bits,pair,rows", [(8192, 1024, 4, False, (17, 31)), (24576, 1024, 4, False, (17, 31)),
                                                (2048, 3840, 4, False, (96,)), (512, 3840, 4, False, (431,)),
                                                (16384, 1024, 4, False, (48,)), (12288, 640, 4, True, (24,)),
                                                (8192, 1024, 8, False, (9, 16, 31)), (16384, 1024, 8, False, (31,)),
                                                (16384, 1088, 8, True, (12, 16))])
def test_graphs_replayed_side_by_side(gpu_lib, n, k, bits, pair, rows):
    import torch

    tri = dev_triple(*_triple(n, k, bits, n + k))
    h = gpu_lib.QuantizedGeGLU(tri, tri, bits=bits) if pair else gpu_lib.QuantizedLinear(*tri, bits=bits)
    for m in rows:
        assert h.scratch_bytes(m) == 0, m
        xs = [dev_x(A.make_activations(m, k, seed=i + m, outliers=True)) for i in range(2)]
        ys = [torch.empty((m, n), dtype=torch.bfloat16, device="cuda") for _ in range(2)]
        cold = torch.cuda.Stream()
        types = G.capture_node_types(cold, lambda: h.forward(xs[0], out=ys[0], stream=cold))
        assert types and all(t == G.KERNEL for t in types), (m, types)
        want = [h.forward(x) for x in xs]
        if not pair:
            got = torch.empty_like(want[0])
            h.forward_noalloc(xs[0], got)
            assert torch.equal(got, want[0]), f"{m} rows: the allocation-free call differs"
        graphs = []
        for x, y in zip(xs, ys):
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=cold):
                for _ in range(8):
                    h.forward(x, out=y)
            graphs.append(g)
        streams = [torch.cuda.Stream(), torch.cuda.Stream()]
        for rep in range(4):
            for y in ys:
                y.zero_()
            torch.cuda.synchronize()
            for g, s in zip(graphs, streams):
                with torch.cuda.stream(s):
                    g.replay()
            torch.cuda.synchronize()
            for y, w in zip(ys, want):
                assert torch.equal(y, w), f"{m} rows, replay {rep}: differs from the eager call"
        del graphs
    h.close()
