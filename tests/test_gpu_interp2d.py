"""2-D interpolation of every stencil width 2m = 2 .. 16 against the oracle: the
lanes of a node's group (2, 4, 8 or 16) pass the dimension-2 weights to one
another, and the last group of a work item, a lone node and groups wider than
the stencil are where that can go wrong.  FP64 rel-l2 <= 1e-12, FP32 <= 1e-5.
"""
import numpy as np
import pytest
import torch

import nfftm
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", range(1, 9))
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32], ids=["f64", "f32"])
def test_widths(m, dtype):
    print(f"interp2d m={m} {dtype}", flush=True)
    N = (30, 37)
    for M, width in ((1, 1.0), (7, 1.0), (301, 0.05), (3001, 1.0)):
        rng = np.random.default_rng([m, M])
        k = width * (rng.random((2, M)) - 0.5)
        p = nfftm.plan_nfft(k, N, m=m, sigma=2.0, precompute=nfftm.LINEAR, dtype=dtype)
        assert p.tile_shape()[1] > 0
        o = O.OraclePlan(k, N, m=m, sigma=2.0, precompute=O.LINEAR)
        g = rng.standard_normal(p.Ntilde) + 1j * rng.standard_normal(p.Ntilde)
        gt = torch.as_tensor(g, dtype=p.dtype, device="cuda")
        want = o.convolve(gt.cpu().numpy().astype(complex))
        got = p.convolve_(gt, torch.empty(M, dtype=p.dtype, device="cuda"))
        assert O.relerr(got.cpu().numpy(), want) < (1e-12 if dtype == torch.float64 else 1e-5), M
