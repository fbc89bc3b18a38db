"""Infinite and NaN node values in FP64 3-D spreading (convolve_transpose!):
only the cells of the node's (2m)^3 footprint take them, as in the oracle's
sums; every other cell keeps its value (FP64 rel-l2 <= 1e-12).

Widths spread by LDS adds (m = 4) and on the matrix cores (m = 5, 6: several
batches and several work items of one tile, whole and ragged grids), values
that are not finite in one part or both.
"""
import numpy as np
import pytest
import torch

import nfftm
import oracle as O

pytestmark = pytest.mark.gpu

INF, NAN = np.inf, np.nan


def same(g, w):
    for a, b in ((g.real, w.real), (g.imag, w.imag)):
        assert np.array_equal(np.isnan(a), np.isnan(b))
        i = np.isinf(b)
        assert np.array_equal(a[i], b[i])
        ok = np.isfinite(b)
        assert ok.any() and np.isfinite(a[ok]).all()
        assert np.linalg.norm(a[ok] - b[ok]) <= 1e-12 * np.linalg.norm(b[ok])


@pytest.mark.parametrize("m", [4, 5, 6])
@pytest.mark.parametrize("N", [(24, 24, 24), (25, 23, 26)], ids=["whole", "ragged"])
@pytest.mark.parametrize("M,width", [(60, 1.0), (2100, 0.02)], ids=["sparse", "crowded"])
def test_footprint_only(m, N, M, width):
    print(f"non-finite spreading m={m} N={N} M={M}", flush=True)
    rng = np.random.default_rng([m, N[0], M])
    k = width * (rng.random((3, M)) - 0.5) + (0.07 if width < 1 else 0.0)
    fh = rng.standard_normal(M) + 1j * rng.standard_normal(M)
    for j, v in ((1, complex(INF, 1.0)), (M // 2, complex(2.0, NAN)), (M - 1, complex(-INF, INF))):
        fh[j] = v
    p = nfftm.plan_nfft(k, N, m=m, sigma=2.0, precompute=nfftm.LINEAR, dtype=torch.float64)
    o = O.OraclePlan(k, N, m=m, sigma=2.0, precompute=O.LINEAR)
    want = o.convolve_transpose(fh)
    assert np.isfinite(want).any() and not np.isfinite(want).all()
    d = torch.as_tensor(fh, device="cuda")
    g = torch.empty(p.Ntilde, dtype=torch.complex128, device="cuda")
    for variant in (0, 1):
        try:
            p.set_tiles(variant, 1024)
        except nfftm.NFFTError:
            continue
        same(p.convolve_transpose_(d, g).cpu().numpy(), want)
