"""Device memory of directional plans that run several slices per launch.

The grids, the scratch areas and the sorted node values (1-D polynomial
windows) of the slices of one launch take at most 512 MiB each; where the
device has less, the plan runs fewer slices per launch.  Results equal the
plan over one slice (FP32 rel-l2 <= 1e-6).
"""
import numpy as np
import pytest
import torch

import nfftm

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def rel(a, b):
    return float(torch.linalg.vector_norm(a - b) / torch.linalg.vector_norm(b))


def check_slices(p, q, S, which):
    f = torch.randn((S, *q.N), dtype=torch.complex64, device="cuda")
    fh = torch.randn((S, q.J), dtype=torch.complex64, device="cuda")
    y, x = p * f, p.H * fh
    for s in which:
        assert rel(y[s], q * f[s]) < 1e-6
        assert rel(x[s], q.H * fh[s]) < 1e-6


def test_sorted_values_are_bounded():
    """80 slices of 10^6 nodes: 8 MB of sorted values each, 67 in 512 MiB."""
    print("slices: sorted values", flush=True)
    rng = np.random.default_rng(1)
    S, N, M = 80, 500, 10 ** 6
    k = rng.random((1, M)) - 0.5
    kw = dict(m=4, sigma=2.0, precompute=nfftm.POLYNOMIAL, dtype=torch.float32)
    q = nfftm.plan_nfft(k, (N,), **kw)
    torch.cuda.empty_cache()
    a = free()
    p = nfftm.plan_nfft(k, (S, N), dims=range(1, 2), **kw)
    assert a - free() < 600 * MIB  # 536 of sorted values, 30 of scratch, 20 of nodes
    check_slices(p, q, S, (0, 66, 67, S - 1))
    c = p.copy()
    check_slices(c, q, S, (0, 66, 67, S - 1))


def test_fewer_slices_where_memory_is_short():
    """A plan that would take 505 MiB of grids and 499 MiB of scratch, created
    and given new nodes with 880 MiB free."""
    print("slices: little memory", flush=True)
    rng = np.random.default_rng(2)
    S, N, M = 64, (600, 600), 100000
    k = rng.random((2, M)) - 0.5
    kw = dict(m=4, sigma=2.0, precompute=nfftm.LINEAR, dtype=torch.float32)
    q = nfftm.plan_nfft(k, N, **kw)
    p0 = nfftm.plan_nfft(k, (S, *N), dims=range(1, 3), **kw)
    check_slices(p0, q, S, (0, S - 1))  # kernels and work arrays are loaded
    torch.cuda.empty_cache()
    fill = []
    keep = 880 * MIB
    try:
        while free() > keep + 16 * MIB:
            fill.append(torch.empty(min(free() - keep, 64 << 30), dtype=torch.uint8, device="cuda"))
        p = nfftm.plan_nfft(k, (S, *N), dims=range(1, 3), **kw)
        p.nodes_(k)
    finally:
        del fill
        torch.cuda.empty_cache()
    check_slices(p, q, S, (0, 20, S - 1))
    k2 = rng.random((2, M)) - 0.5
    q.nodes_(k2)
    p.nodes_(k2)
    check_slices(p, q, S, (0, 20, S - 1))
