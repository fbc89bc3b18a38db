"""FFT passes with per-plan radices (k_mixfft.hip) at the ends of their range,
against the whole-grid rocFFT stage (FP64 rel-l2 <= 1e-13, FP32 <= 2e-6).

Lines of one pass (16 points) and the longest ones: 8190 points of a 1-D FP32
grid and 4096 of an FP64 one (a whole workgroup on one line), strided and
dimension-1 lines of up to 2048 points beside short axes, in 2-D and 3-D.  The
plans are directional with one slice, so that forward and adjoint of both
precisions take the passes.  Toeplitz products on both sides of the sizes whose
last-dimension pass (two lines' LDS areas) no longer fits the LDS, and of those
whose lines are taken without radix 16, against FFTs of the padded image in FP64.
"""
import numpy as np
import pytest
import torch

import nfftm
import oracle as O
from nfftm import tools

pytestmark = pytest.mark.gpu

F32, F64 = torch.float32, torch.float64
BOTH = (F64, F32)

CASES = [
    ((8, 9), BOTH),             # 16 = one pass, beside 18
    ((9, 8), BOTH),
    ((8, 9, 8), BOTH),
    ((4095,), (F32,)),          # 8190 = 2 3^2 5 7 13
    ((4096,), (F32,)),          # 8192, the longest
    ((4080,), (F32,)),          # 8160 = 2^5 3 5 17: rocFFT
    ((4032,), (F32,)),          # 8064 = 2^7 3^2 7
    ((2048,), (F64,)),          # 4096, the longest
    ((2028,), (F64,)),          # 4056 = 2^3 3 13^2
    ((2016,), (F64,)),          # 4032
    ((2000,), BOTH),
    ((990, 12), BOTH),          # 1980 = 2^2 3^2 5 11 along dimension 2
    ((12, 990), BOTH),          # and along dimension 1
    ((1024, 10), BOTH),         # 2048, the longest strided line
    ((10, 1024), BOTH),
    ((1001, 9), BOTH),          # 2002 = 2 7 11 13
    ((1020, 9), BOTH),          # 2040 = 2^3 3 5 17: rocFFT
    ((1000, 33), BOTH),
    ((990, 9, 10), BOTH),       # along dimension 3
    ((9, 1024, 10), BOTH),
    ((9, 10, 1014), BOTH),      # 2028 along dimension 1
]


def rel(a, b):
    return O.relerr(a.cpu().numpy(), b.cpu().numpy())


@pytest.mark.parametrize("N,dtype", [(N, t) for N, ts in CASES for t in ts],
                         ids=[f"{'x'.join(map(str, N))}-{'f64' if t == F64 else 'f32'}" for N, ts in CASES for t in ts])
def test_lines(N, dtype):
    print(f"lines N={N} {dtype}", flush=True)
    rng = np.random.default_rng([len(N), sum(N)])
    D, M = len(N), 3000
    k = rng.random((D, M)) - 0.5
    kw = dict(m=3, sigma=2.0, precompute=nfftm.LINEAR, dtype=dtype, dims=range(1, D + 1))
    p = nfftm.plan_nfft(k, (1, *N), **kw)
    q = nfftm.plan_nfft(k, (1, *N), rocfft=True, **kw)
    cd = torch.complex128 if dtype == F64 else torch.complex64
    tol = 1e-13 if dtype == F64 else 2e-6
    for _ in range(2):
        f = torch.as_tensor(rng.standard_normal((1, *N)) + 1j * rng.standard_normal((1, *N)), dtype=cd, device="cuda")
        fh = torch.as_tensor(rng.standard_normal((1, M)) + 1j * rng.standard_normal((1, M)), dtype=cd, device="cuda")
        y, yq = p * f, q * f
        assert rel(p.tmpVec, q.tmpVec) < tol
        assert rel(y, yq) < tol
        assert rel(p.H * fh, q.H * fh) < tol


# Lines of 2 n points along the last (first Python) dimension.  Short rest axes
# give the fewest lines per workgroup (FP64 2, FP32 4), the long ones 8 or 4.
TOEP = [(n, r) for r in [(9,), (6, 5)] for n in (500, 693, 728, 735, 924, 936, 1024)]
TOEP += [(128, (128,)), (48, (56,)), (8, (64,)), (128, (129,))]  # up to 256^2 points and above
TOEP += [(n, (40, 60)) for n in (264, 273, 462, 468, 528, 539, 546, 600, 1024)]


@pytest.mark.parametrize("n,rest", TOEP, ids=["x".join(map(str, (n, *r))) for n, r in TOEP])
@pytest.mark.parametrize("dtype", [torch.complex128, torch.complex64], ids=["f64", "f32"])
def test_toeplitz_long_lines(n, rest, dtype):
    shape = (n, *rest)
    print(f"toeplitz {shape} {dtype}", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    lam = torch.randn(tuple(2 * s for s in shape), dtype=dtype, device="cuda", generator=g)
    t = tools.Toeplitz(shape, dtype)
    y = torch.randn(shape, dtype=dtype, device="cuda", generator=g)
    crop = tuple(slice(0, s) for s in shape)
    pad = torch.zeros(lam.shape, dtype=torch.complex128, device="cuda")
    pad[crop] = y.to(torch.complex128)
    want = torch.fft.ifftn(torch.fft.fftn(pad) * lam.to(torch.complex128))[crop]
    got = tools.convolveToeplitzKernel_(y, lam, t)
    assert ((got - want).norm() / want.norm()).item() < (1e-13 if dtype == torch.complex128 else 2e-6)
