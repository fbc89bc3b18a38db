"""Interpolation on work items of every number of steps: the lanes of a node's
group keep the results of up to G steps (G = 2, 4, 8, 16; FP32 four) and store
them together, so a lone step, a whole round, one more and items of several rounds are where a node
could be left out or written twice.  Against the oracle: FP64 rel-l2 <= 1e-12,
FP32 <= 1e-5; density weights (their update is made at the same place) <= 1e-10
and 1e-5.
"""
import numpy as np
import pytest
import torch

import nfftm
import oracle as O
from nfftm import tools as T

pytestmark = pytest.mark.gpu

# nodes of one tile: a step of a workgroup of 512 takes 512 / G of them
COUNTS = (1, 31, 32, 33, 64, 65, 255, 256, 257, 511, 512, 513, 1024, 1025, 2048, 2049, 4097)


def tol(dtype):
    return 1e-12 if dtype == torch.float64 else 1e-5


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("m", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("D", [1, 2])
def test_steps(D, m, dtype):
    print(f"interp steps D={D} m={m} {dtype}", flush=True)
    N = (600,) if D == 1 else (40, 44)
    rng = np.random.default_rng([D, m])
    for M in COUNTS:
        k = 0.1 + 0.01 * rng.random((D, M))  # one tile, or two at its border
        p = nfftm.plan_nfft(k, N, m=m, sigma=2.0, precompute=nfftm.LINEAR, dtype=dtype)
        assert p.tile_shape()[1] > 0
        o = O.OraclePlan(k, N, m=m, sigma=2.0, precompute=O.LINEAR)
        g = rng.standard_normal(p.Ntilde) + 1j * rng.standard_normal(p.Ntilde)
        gt = torch.as_tensor(g, dtype=p.dtype, device="cuda")
        got = p.convolve_(gt, torch.full((M,), float("nan"), dtype=p.dtype, device="cuda"))
        assert O.relerr(got.cpu().numpy(), o.convolve(gt.cpu().numpy().astype(complex))) < tol(dtype), M


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("M", [1, 65, 512, 513, 4097])
def test_sdc_steps(M, dtype):
    print(f"sdc steps M={M} {dtype}", flush=True)
    rng = np.random.default_rng(M)
    k = 0.1 + 0.05 * rng.random((2, M))
    p = nfftm.plan_nfft(k, (40, 44), m=4, sigma=2.0, precompute=nfftm.LINEAR, dtype=dtype)
    w = T.sdc(p, iters=4).cpu().numpy()
    orc = O.OraclePlan(k, (40, 44), m=4, sigma=2.0, precompute=O.LINEAR)
    assert O.relerr(w, O.sdc(orc, iters=4)) < (1e-10 if dtype == torch.float64 else 1e-5)


def test_batch_steps():
    """The same items in a batch."""
    print("batch steps", flush=True)
    rng = np.random.default_rng(5)
    plans = []
    for M in (1, 65, 513, 2049):
        k = 0.1 + 0.05 * rng.random((2, M))
        plans.append(nfftm.plan_nfft(k, (40, 44), m=4, sigma=2.0, precompute=nfftm.LINEAR))
    b = nfftm.BatchPlan(plans, autotune=False)
    fs = [torch.randn((40, 44), dtype=torch.complex128, device="cuda") for _ in plans]
    for y, p, f in zip(b.forward(fs), plans, fs):
        assert O.relerr(y.cpu().numpy(), (p * f).cpu().numpy()) < 1e-13
