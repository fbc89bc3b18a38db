"""Directional plans that run several slices per launch, against the same
plan's slices one at a time.

The kernels find a slice's image, node values, grid and scratch by its index;
the cases cover slices before, after and on both sides of the transformed axes,
the FFT stages (power-of-two passes, per-plan radices, rocFFT), 1-D plans with
the window evaluated in the kernel and with records, more slices than one
launch takes (256), and the grid left by the last slice.  FP64 rel-l2 <= 1e-13
(spreading sums in LDS are not ordered), FP32 <= 1e-6.
"""
import numpy as np
import pytest
import torch

import nfftm
import oracle as O

pytestmark = pytest.mark.gpu

# N, dims, M, precompute
CASES = [
    ((5, 16, 32), (1, 2), 900, nfftm.LINEAR),       # power-of-two grid, slices first
    ((16, 16, 7), (0, 1), 900, nfftm.POLYNOMIAL),   # slices last
    ((3, 20, 18, 4), (1, 2), 900, nfftm.LINEAR),    # both sides, 40 x 36
    ((3, 17, 19, 2), (1, 2), 900, nfftm.LINEAR),    # 34 x 38: rocFFT
    ((6, 500), (1, 1), 1500, nfftm.TENSOR),         # 1-D, window in the kernel
    ((500, 6), (0, 0), 1500, nfftm.LINEAR),         # 1-D, records
    ((300, 15, 14), (1, 2), 300, nfftm.LINEAR),     # more than one launch
    ((7, 10, 40, 3), (2, 2), 700, nfftm.POLYNOMIAL),
]


@pytest.mark.parametrize("N,dims,M,pre", CASES, ids=["x".join(map(str, c[0])) for c in CASES])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32], ids=["f64", "f32"])
def test_slices_together(N, dims, M, pre, dtype):
    print(f"slices N={N} dims={dims} pre={pre} {dtype}", flush=True)
    rng = np.random.default_rng([len(N), M])
    ax = range(dims[0], dims[1] + 1)
    D = len(ax)
    k = rng.random((D, M)) - 0.5
    kw = dict(m=4, sigma=2.0, precompute=pre, dtype=dtype)
    p = nfftm.plan_nfft(k, N, dims=ax, **kw)
    q = nfftm.plan_nfft(k, tuple(N[a] for a in ax), **kw)
    cd = torch.complex128 if dtype == torch.float64 else torch.complex64
    tol = 1e-13 if dtype == torch.float64 else 1e-6
    for kk in (k, rng.random((D, M // 2)) - 0.5):
        p.nodes_(kk)
        q.nodes_(kk)
        f = torch.as_tensor(rng.standard_normal(N) + 1j * rng.standard_normal(N), dtype=cd, device="cuda")
        fh = torch.as_tensor(rng.standard_normal(p.NOut) + 1j * rng.standard_normal(p.NOut), dtype=cd, device="cuda")
        y, g = p * f, p.tmpVec.clone()
        x = p.H * fh
        B, A = int(np.prod(N[:dims[0]], dtype=int)), int(np.prod(N[dims[1] + 1:], dtype=int))
        fs = f.reshape(B, *q.N, A)
        hs = fh.reshape(B, q.J, A)
        ys = torch.stack([torch.stack([q * fs[b, ..., a].contiguous() for a in range(A)], -1) for b in range(B)])
        glast = q.tmpVec.clone()
        xs = torch.stack([torch.stack([q.H * hs[b, :, a].contiguous() for a in range(A)], -1) for b in range(B)])
        torch.cuda.synchronize()
        assert O.relerr(y.reshape(ys.shape).cpu().numpy(), ys.cpu().numpy()) < tol
        assert O.relerr(x.reshape(xs.shape).cpu().numpy(), xs.cpu().numpy()) < tol
        assert O.relerr(g.cpu().numpy(), glast.cpu().numpy()) < tol
    c = p.copy()
    assert O.relerr((c * f).cpu().numpy(), (p * f).cpu().numpy()) < tol
