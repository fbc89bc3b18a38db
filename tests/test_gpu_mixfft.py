"""Pruned FFT passes with per-plan radices (k_mixfft.hip) against the
whole-grid rocFFT stage and the oracle.

Grids that are not powers of two: FP64 rel-l2 <= 1e-13 between the two paths
and <= 1e-12 against the CPU oracle; FP32 <= 2e-6 between the paths (forward
transforms of FP32 plans that are not directional run rocFFT themselves).  The
sizes cover every radix of the list, lines of two to four passes, few and many
lines per workgroup, ragged chunks of lines and a grid that stays with rocFFT
(302 = 2 151); the ends of the range are in test_gpu_mixfft_lines.py.
"""
import numpy as np
import pytest
import torch

import nfftm
import oracle as O

pytestmark = pytest.mark.gpu


def rel(a, b):
    return O.relerr(a.detach().cpu().numpy(), b.detach().cpu().numpy() if isinstance(b, torch.Tensor) else b)


def crandn(rng, shape):
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


# (N in C order, sigma)
CASES = [
    ((9,), 2.0),              # Nt = 18 = 9 2
    ((63,), 2.0),             # 126 = 9 7 2
    ((2000,), 2.0),           # 4000, four passes
    ((143,), 2.0),            # 286 = 2 11 13
    ((13, 11), 2.0),          # 26 = 2 13, 22 = 2 11
    ((10, 24), 2.0),          # 20, 48
    ((75, 96), 2.0),          # 150, 192
    ((250, 37), 1.21),        # 302 = 2 151 beside 44: rocFFT for both
    ((320, 45), 2.0),         # 640, 90
    ((81, 147), 2.0),         # 162, 294 = 2 3 7 7
    ((700, 20), 2.0),         # 1400 = 2^3 5^2 7
    ((9, 10, 12), 2.0),       # 18, 20, 24
    ((25, 18, 21), 2.0),      # 50, 36, 42
    ((30, 33, 26), 2.0),      # 60, 66 = 6 11, 52 = 4 13
    ((48, 50, 45), 2.0),      # 96, 100, 90
]


@pytest.mark.parametrize("N,sigma", CASES, ids=["x".join(map(str, c[0])) for c in CASES])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32], ids=["f64", "f32"])
def test_mix_matches_rocfft(N, sigma, dtype):
    print(f"mix N={N} sigma={sigma:.4f} dtype={dtype}", flush=True)
    rng = np.random.default_rng([len(N), sum(N), dtype == torch.float64])
    M = 3000 if np.prod(N) < 1e5 else 40000
    k = rng.random((len(N), M)) - 0.5
    kw = dict(m=4, sigma=sigma, precompute=nfftm.LINEAR, dtype=dtype)
    p = nfftm.plan_nfft(k, N, **kw)
    q = nfftm.plan_nfft(k, N, rocfft=True, **kw)
    cd = torch.complex128 if dtype == torch.float64 else torch.complex64
    tol = 1e-13 if dtype == torch.float64 else 2e-6
    for it in range(2):
        f = torch.as_tensor(crandn(rng, N), dtype=cd, device="cuda")
        fh = torch.as_tensor(crandn(rng, M), dtype=cd, device="cuda")
        y, yq = p * f, q * f
        g, gq = p.tmpVec.clone(), q.tmpVec.clone()
        x, xq = p.H * fh, q.H * fh
        torch.cuda.synchronize()
        assert rel(g, gq) < tol
        assert rel(y, yq) < tol
        assert rel(x, xq) < tol
    if dtype == torch.float64 and np.prod(N) <= 8192:
        orc = O.OraclePlan(k, N, m=4, sigma=sigma, precompute=O.LINEAR)
        assert rel(y, orc.forward(f.cpu().numpy())) < 1e-12
        assert rel(x, orc.adjoint(fh.cpu().numpy())) < 1e-12


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32], ids=["f64", "f32"])
def test_mix_slices(dtype):
    """A directional plan on such a grid: strided image slices on either side
    of the transformed axes."""
    rng = np.random.default_rng(3)
    N, dims = (3, 20, 15, 5), range(1, 3)
    k = rng.random((2, 700)) - 0.5
    kw = dict(m=4, sigma=2.0, precompute=nfftm.LINEAR, dtype=dtype)
    p = nfftm.plan_nfft(k, N, dims=dims, **kw)
    q = nfftm.plan_nfft(k, N, dims=dims, rocfft=True, **kw)
    cd = torch.complex128 if dtype == torch.float64 else torch.complex64
    tol = 1e-13 if dtype == torch.float64 else 2e-6
    f = torch.as_tensor(crandn(rng, N), dtype=cd, device="cuda")
    fh = torch.as_tensor(crandn(rng, p.NOut), dtype=cd, device="cuda")
    assert rel(p * f, q * f) < tol
    assert rel(p.H * fh, q.H * fh) < tol
