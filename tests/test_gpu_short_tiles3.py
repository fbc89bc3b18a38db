"""Tile edge along dimension 3 of FP64 plans with 2m = 10: 8 x 8 x 16 cells, or
8^3 where the grid is shorter than the long tile's padded edge (25 cells), has
the volume of fewer than 1024 long tiles, or the plan is made for no more nodes
than long tiles.

Every grid that holds the cubic tile's padded edge (17 cells) is tiled, and
forward and adjoint equal the oracle (FP64 rel-l2 <= 1e-12) on both sides of
each line, on thin nodes and on crowded ones.
"""
import numpy as np
import pytest
import torch

import nfftm
import oracle as O

pytestmark = pytest.mark.gpu


def plan(N, M, m=5, dtype=torch.float64, crowded=False):
    rng = np.random.default_rng([sum(N), M])
    k = rng.random((3, M)) - 0.5
    if crowded:
        k *= 0.15
    return k, nfftm.plan_nfft(k, N, m=m, sigma=2.0, precompute=nfftm.LINEAR, dtype=dtype)


# (N in C order, tile in C order: dimension 3 first)
CASES = [
    ((9, 20, 22), (8, 8, 8)),   # Nt[2] = 18, one cell more than the padded edge
    ((12, 24, 9), (8, 8, 8)),   # 24, one short of the long tile's
    ((13, 24, 20), (8, 8, 8)),  # 26, few tiles
    ((24, 24, 24), (8, 8, 8)),
]


@pytest.mark.parametrize("N,tile", CASES, ids=["x".join(map(str, c[0])) for c in CASES])
@pytest.mark.parametrize("crowded", [False, True], ids=["thin", "crowded"])
def test_short_tile(N, tile, crowded):
    print(f"short tile N={N} crowded={crowded}", flush=True)
    M = 2500 if crowded else 400
    k, p = plan(N, M, crowded=crowded)
    assert p.tile_shape()[0] == tile
    rng = np.random.default_rng(M)
    f = rng.standard_normal(N) + 1j * rng.standard_normal(N)
    fh = rng.standard_normal(M) + 1j * rng.standard_normal(M)
    o = O.OraclePlan(k, N, m=5, sigma=2.0, precompute=O.LINEAR)
    want, wantH = o.forward(f), o.adjoint(fh)
    ft, fht = torch.as_tensor(f, device="cuda"), torch.as_tensor(fh, device="cuda")

    def check():
        assert O.relerr((p * ft).cpu().numpy(), want) < 1e-12
        assert O.relerr((p.H * fht).cpu().numpy(), wantH) < 1e-12

    check()
    for variant in (1, 0):
        for nt in (512, 1024):
            try:
                p.set_tiles(variant, nt)
            except nfftm.NFFTError:
                continue
            check()
    assert p.tile_shape()[0] == tile
    p.tune()
    check()


def test_lines():
    """1024 long tiles: 16 x 8 x 8 of them; one fewer along dimension 1, or
    another width or precision: the tile of that side."""
    _, p = plan((64, 32, 32), 300)   # Nt = 128 x 64 x 64: 8 * 8 * 8 tiles
    assert p.tile_shape()[0] == (8, 8, 8)
    k, p = plan((64, 64, 64), 3000)  # 16 * 16 * 8
    assert p.tile_shape()[0] == (16, 8, 8)
    f = torch.randn((64, 64, 64), dtype=torch.complex128, device="cuda")
    fh = torch.randn(3000, dtype=torch.complex128, device="cuda")
    q = nfftm.plan_nfft(k, (64, 64, 64), m=5, sigma=2.0, precompute=nfftm.LINEAR, sparse_matrix=True)
    assert O.relerr((p * f).cpu().numpy(), (q * f).cpu().numpy()) < 1e-13
    assert O.relerr((p.H * fh).cpu().numpy(), (q.H * fh).cpu().numpy()) < 1e-13
    for m, dtype in ((4, torch.float64), (6, torch.float64), (5, torch.float32)):
        assert plan((24, 24, 24), 300, m, dtype)[1].tile_shape()[1] == 1024
    _, p = plan((8, 30, 30), 300)    # 16 cells: node-parallel, as before
    assert p.tile_shape()[0] == (0, 0, 0)


@pytest.mark.parametrize("N,n", [((64, 64, 64), 2048), ((50, 50, 53), 1035)], ids=["whole", "ragged"])
def test_few_nodes(N, n):
    """Up to n nodes, n the volume of the grid in long tiles: the cubic tile, also
    on power-of-two grids (separate fold); one more: the long one.  nodes!
    keeps the tile, copy and set_tiles choose for the nodes there are."""
    print(f"short tile, few nodes N={N}", flush=True)

    def check(p, k):
        M = k.shape[1]
        q = nfftm.plan_nfft(k, N, m=5, sigma=2.0, precompute=nfftm.LINEAR, sparse_matrix=True)
        f = torch.randn(N, dtype=torch.complex128, device="cuda")
        fh = torch.randn(M, dtype=torch.complex128, device="cuda")
        assert O.relerr((p * f).cpu().numpy(), (q * f).cpu().numpy()) < 1e-13
        assert O.relerr((p.H * fh).cpu().numpy(), (q.H * fh).cpu().numpy()) < 1e-13

    ka, a = plan(N, n)
    kb, b = plan(N, n + 1)
    assert a.tile_shape()[0] == (8, 8, 8) and b.tile_shape()[0] == (16, 8, 8)
    check(a, ka)
    check(b, kb)
    a.nodes_(kb)
    b.nodes_(ka)
    assert a.tile_shape()[0] == (8, 8, 8) and b.tile_shape()[0] == (16, 8, 8)
    check(a, kb)
    check(b, ka)
    c = a.copy()
    assert c.tile_shape()[0] == (16, 8, 8)
    check(c, kb)
    b.set_tiles(0, 1024)
    assert b.tile_shape()[0] == (8, 8, 8)
    check(b, ka)
