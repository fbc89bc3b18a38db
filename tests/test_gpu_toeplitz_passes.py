"""Toeplitz products on the pruned line passes (pad, product and crop fused)
against FFTs of the padded image in torch: even, odd and ragged sizes in 2-D and
3-D, a size with a prime factor the passes are not built for (rocFFT), and
repeated products with one object.  FP64 rel-l2 <= 1e-13, FP32 <= 2e-6.
"""
import pytest
import torch

from nfftm import tools

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(16, 20), (33, 15), (256, 256), (9, 150), (12, 10, 14), (8, 33, 9), (17, 19), (40,)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("dtype", [torch.complex128, torch.complex64], ids=["f64", "f32"])
def test_product(shape, dtype):
    print(f"toeplitz passes {shape} {dtype}", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(len(shape))
    lam = torch.randn(tuple(2 * n for n in shape), dtype=dtype, device="cuda", generator=g)
    t = tools.Toeplitz(shape, dtype)
    y = torch.randn(shape, dtype=dtype, device="cuda", generator=g)
    for _ in range(3):
        pad = torch.zeros(lam.shape, dtype=torch.complex128, device="cuda")
        crop = tuple(slice(0, n) for n in shape)
        pad[crop] = y.to(torch.complex128)
        want = torch.fft.ifftn(torch.fft.fftn(pad) * lam.to(torch.complex128))[crop]
        got = tools.convolveToeplitzKernel_(y, lam, t)
        assert got is y
        err = ((got - want).norm() / want.norm()).item()
        assert err < (1e-13 if dtype == torch.complex128 else 2e-6)
