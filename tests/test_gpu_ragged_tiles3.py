"""3-D spreading on grids that are no multiple of the tile, and on crowded
tiles, against the oracle.

The halo/interior block layout of the slots holds for a partial last tile
(its right halo follows its own cells) as long as that tile has at least m
cells; below that the per-dimension pieces remain.  Tiles of several work
items (more than 1024 nodes) are summed into one slot before the fold.  FP64
rel-l2 <= 1e-12 against the oracle; FP32 <= 1e-5, the bar of every FP32 result.
"""
import numpy as np
import pytest
import torch

import nfftm
import oracle as O

pytestmark = pytest.mark.gpu

# N in C order, m: FP32 tiles are 16 x 16 x 16 or 16 x 16 x 8 cells, FP64 8 to 12
CASES = [
    ((13, 15, 20), 2),   # 26, 30, 40 points
    ((17, 20, 13), 3),   # 34 = 2 16 + 2 (FP32: last tile below m), 40, 26
    ((25, 22, 19), 4),   # 50, 44, 38
    ((24, 16, 21), 4),   # 48 and 32 whole, 42 ragged
    ((20, 24, 23), 5),
    ((27, 25, 26), 6),
]


@pytest.mark.parametrize("N,m", CASES, ids=["x".join(map(str, c[0])) + f"-m{c[1]}" for c in CASES])
@pytest.mark.parametrize("nodes", ["uniform", "crowded", "edges"])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32], ids=["f64", "f32"])
def test_ragged_spreading(N, m, nodes, dtype):
    print(f"ragged3 N={N} m={m} nodes={nodes} {dtype}", flush=True)
    rng = np.random.default_rng([m, sum(N), len(nodes)])
    M = 4000
    k = rng.random((3, M)) - 0.5
    if nodes == "crowded":  # most nodes in two tiles: several work items each
        k[:, :2200] = 0.01 * k[:, :2200] + 0.1
        k[:, 2200:3700] *= 0.02
    if nodes == "edges":    # across the periodic border, where the partial tiles are
        k = np.where(k < 0, -0.5 + 0.1 * (k + 0.5), 0.5 - 0.1 * (0.5 - k))
    kw = dict(m=m, sigma=2.0, precompute=nfftm.LINEAR, dtype=dtype)
    p = nfftm.plan_nfft(k, N, **kw)
    cd = torch.complex128 if dtype == torch.float64 else torch.complex64
    fh = rng.standard_normal(M) + 1j * rng.standard_normal(M)
    if dtype == torch.float32:
        fh = fh.astype(np.complex64).astype(np.complex128)
    x = (p.H * torch.as_tensor(fh, dtype=cd, device="cuda")).cpu().numpy()
    o = O.OraclePlan(k, N, m=m, sigma=2.0, precompute=O.LINEAR)
    assert O.relerr(x, o.adjoint(fh)) < (1e-12 if dtype == torch.float64 else 1e-5)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32], ids=["f64", "f32"])
def test_crowded_then_even(dtype):
    """Crowded tiles on a power-of-two grid (separate fold), then nodes! to an
    even spread (the fold fused into the first FFT pass) and back, against a
    plan that always folds separately."""
    rng = np.random.default_rng(8)
    N, M = (64, 64, 64), 30000
    k = np.concatenate([0.02 * (rng.random((3, M // 2)) - 0.5), rng.random((3, M // 2)) - 0.5], axis=1)
    kw = dict(m=4, sigma=2.0, precompute=nfftm.LINEAR, dtype=dtype)
    p = nfftm.plan_nfft(k, N, **kw)
    q = nfftm.plan_nfft(k, N, fused_fold=False, **kw)
    cd = torch.complex128 if dtype == torch.float64 else torch.complex64
    fh = torch.as_tensor(rng.standard_normal(M) + 1j * rng.standard_normal(M), dtype=cd, device="cuda")
    tol = 1e-13 if dtype == torch.float64 else 1e-6
    for kk in (k, rng.random((3, M)) - 0.5, k):
        p.nodes_(kk)
        q.nodes_(kk)
        a, b = p.H * fh, q.H * fh
        assert O.relerr(a.cpu().numpy(), b.cpu().numpy()) < tol
