"""Node gradients of FP32 plans on grids that are not powers of two.

The node gradient is FP64 also where the plan is FP32; it is gathered from the
grid of the forward transform, and carries that grid's FP32 digits.  The FFT
stage of the forward transform of an FP32 plan is therefore fixed on these
grids: every route to the gradient (grad_nodes, grad_nodes_grid on the plan's
grid, the rrule and the torch function) equals that of a plan on the
whole-grid FFT bit for bit.  Against the oracle's FP64 gradient: 1e-5.
"""
import numpy as np
import pytest
import torch

import nfftm
import oracle as O
from nfftm import autograd as AD

pytestmark = pytest.mark.gpu

# Nt = 180 x 216, 128 x 208 (one dimension a power of two), 286 = 2 11 13,
# 60 x 66 x 52, 302 = 2 151 (no line passes)
CASES = [(90, 108), (64, 104), (143,), (30, 33, 26), (151, 20)]


@pytest.mark.parametrize("N", CASES, ids=lambda v: "x".join(map(str, v)))
@pytest.mark.parametrize("pre", [nfftm.LINEAR, nfftm.POLYNOMIAL], ids=["linear", "polynomial"])
def test_fp32_gradient_equals_whole_grid_fft(N, pre):
    print(f"fp32 node gradient N={N} pre={pre}", flush=True)
    rng = np.random.default_rng([len(N), sum(N), pre])
    D, M = len(N), 1500
    k = rng.random((D, M)) - 0.5
    kw = dict(m=4, sigma=2.0, precompute=pre, dtype=torch.float32)
    p, q = nfftm.plan_nfft(k, N, **kw), nfftm.plan_nfft(k, N, rocfft=True, **kw)
    f = rng.standard_normal(N) + 1j * rng.standard_normal(N)
    yb = rng.standard_normal(M) + 1j * rng.standard_normal(M)
    ft = torch.as_tensor(f, dtype=torch.complex64, device="cuda")
    ybt = torch.as_tensor(yb, dtype=torch.complex64, device="cuda")
    want = q.grad_nodes(ft, ybt)
    assert want.dtype == torch.float64
    assert torch.equal(p.grad_nodes(ft, ybt), want)
    y = p * ft
    assert torch.equal(y, q * ft)
    assert torch.equal(p.grad_nodes_grid(p.tmpVec, ybt), want)
    _, pullback = AD.rrule_nfft(k, ft, plan=p)
    assert torch.equal(pullback(ybt)[0], want)
    kt = torch.as_tensor(k, device="cuda").requires_grad_(True)
    kbar, = torch.autograd.grad(AD.nfft(kt, ft, plan=p), (kt,), ybt)
    assert torch.equal(kbar, want)
    orc = O.OraclePlan(k, N, m=4, sigma=2.0, precompute=pre if pre == nfftm.LINEAR else O.POLYNOMIAL)
    ref = orc.grad_nodes(ft.cpu().numpy().astype(complex), ybt.cpu().numpy().astype(complex))
    assert O.relerr(want.cpu().numpy(), ref) < 1e-5
