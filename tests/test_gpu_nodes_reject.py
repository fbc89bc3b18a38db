"""nodes! with a node outside [-1/2, 1/2] or NaN (checkNodes, src/utils.jl:46-55),
found by the binning kernels on the device (by a kernel of its own, or on the
host, for node-parallel plans): ArgumentError, and the plan goes on with its old
nodes (forward bit for bit, adjoint FP32 rel-l2 <= 1e-6); a following nodes!
with valid nodes and another M equals a fresh plan.

Both layouts of the entry point (rows, as the Python wrapper passes them, and
Julia's D x M), the bad coordinate first, in the middle and last, in each
dimension; tiled plans of few tiles (histogram in LDS) and of more than 16,384,
1-D, 2-D and 3-D, and a node-parallel plan.  The closed ends are accepted.
"""
import ctypes

import numpy as np
import pytest
import torch

import nfftm

pytestmark = pytest.mark.gpu

# N, M, tiled
CASES = {
    "line": ((600,), 700, True),
    "image": ((64, 48), 900, True),
    "manytiles": ((1100, 1200), 3000, True),  # 138 x 150 tiles of 16^2
    "volume": ((24, 20, 28), 800, True),
    "nodeparallel": ((8, 7), 500, False),      # looked at on the host
    "nodeparallel_many": ((8, 7), 5000, False),
}


def rel(a, b):
    return float(torch.linalg.vector_norm(a - b) / torch.linalg.vector_norm(b))


def julia_nodes(p, k):
    """nfftm_nodes: Julia's D x M matrix (node after node, dimensions reversed)."""
    kj = np.ascontiguousarray(k[::-1].T, dtype=np.float64)
    torch.cuda.synchronize()
    rc = p._lib.nfftm_nodes(p._handle, kj.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), k.shape[1])
    if rc:
        raise nfftm.ArgumentError(p._lib.nfftm_last_error().decode()) if rc == 1 else nfftm.NFFTError(str(rc))


@pytest.mark.parametrize("entry", ["rows", "julia"])
@pytest.mark.parametrize("case", CASES)
def test_bad_node_is_refused(case, entry):
    N, M, tiled = CASES[case]
    print(f"bad nodes {case} {entry}", flush=True)
    rng = np.random.default_rng([M, len(case)])
    D = len(N)
    kw = dict(m=4, sigma=2.0, precompute=nfftm.LINEAR, dtype=torch.float32)
    k = rng.random((D, M)) - 0.5
    k[:, 0], k[:, 1] = -0.5, 0.5
    p = nfftm.plan_nfft(k, N, **kw)
    assert (p.tile_shape()[1] > 0) == tiled
    set_nodes = p.nodes_ if entry == "rows" else lambda kk: julia_nodes(p, kk)
    f = torch.randn(N, dtype=torch.complex64, device="cuda")
    fh = torch.randn(M, dtype=torch.complex64, device="cuda")
    y, x = p * f, p.H * fh
    for bad in (0.6, -0.51, np.nan, np.inf):
        for d in range(D):
            for j, Mb in ((0, M), (M // 2, M), (M + 99, M + 100)):  # fewer, as many and more nodes
                kb = rng.random((D, Mb)) - 0.5
                kb[d, j] = bad
                with pytest.raises(nfftm.ArgumentError):
                    set_nodes(kb)
                assert p.J == M
        assert torch.equal(p * f, y)
        assert rel(p.H * fh, x) < 1e-6
    k2 = rng.random((D, M + 50)) - 0.5
    k2[:, -1], k2[:, 0] = 0.5, -0.5
    set_nodes(k2)
    p._read_sizes()
    q = nfftm.plan_nfft(k2, N, **kw)
    fh2 = torch.randn(M + 50, dtype=torch.complex64, device="cuda")
    assert torch.equal(p * f, q * f)
    assert rel(p.H * fh2, q.H * fh2) < 1e-6
