"""FP64 3-D spreading against the oracle: on the matrix cores from 2m = 10 on
(k_spread3d: two row tiles along z, whole and partial column tiles), by LDS
adds below.

Every stencil width 2m = 2 .. 16, both tile geometries and both workgroup
sizes, nodes that fill groups of four exactly, leave one over, or share one
cell, tiles of one node, items of several batches and several items; FP64
rel-l2 <= 1e-12.
"""
import numpy as np
import pytest
import torch

import nfftm
import oracle as O

pytestmark = pytest.mark.gpu


def check(k, N, m, **kw):
    rng = np.random.default_rng(len(k[0]))
    p = nfftm.plan_nfft(k, N, m=m, sigma=2.0, precompute=nfftm.LINEAR, dtype=torch.float64, **kw)
    o = O.OraclePlan(k, N, m=m, sigma=2.0, precompute=O.LINEAR)
    fh = rng.standard_normal(k.shape[1]) + 1j * rng.standard_normal(k.shape[1])
    want = o.adjoint(fh)
    d = torch.as_tensor(fh, dtype=torch.complex128, device="cuda")
    assert O.relerr((p.H * d).cpu().numpy(), want) < 1e-12
    return p, d, want


@pytest.mark.parametrize("m", range(1, 9))
@pytest.mark.parametrize("nodes", ["sparse", "dense"])
def test_widths(m, nodes):
    print(f"spread3d m={m} {nodes}", flush=True)
    rng = np.random.default_rng([m, len(nodes)])
    N = (20, 17, 18)
    if nodes == "sparse":
        k = rng.random((3, 301)) - 0.5
    else:  # a few crowded tiles: several batches of an item, items of 1024
        k = 0.2 * (rng.random((3, 3001)) - 0.5) + 0.1
    p, d, want = check(k, N, m)
    for variant in (0, 1):
        for nt in (512, 1024):
            try:
                p.set_tiles(variant, nt)
            except nfftm.NFFTError:
                continue  # no such geometry for this width
            assert O.relerr((p.H * d).cpu().numpy(), want) < 1e-12, (variant, nt)


@pytest.mark.parametrize("M", [1, 3, 4, 5, 255, 256, 257, 1024, 1029])
def test_counts(M):
    """One tile with M nodes: groups, batches and items that end anywhere."""
    rng = np.random.default_rng(M)
    for spread in (0.0, 0.04):
        k = 0.11 + spread * (rng.random((3, M)) - 0.5)
        for m in (4, 5, 6):
            check(k, (24, 24, 24), m)
