"""nodes! on a plan while a batch that holds it is still running on another
stream: nodes! rewrites the plan's node arrays in place, so it waits for the
batch first (as it does for set_tiles and tune, which bin the nodes again).
The batch's outputs are those of the old nodes: forward bit for bit (the
interpolation is deterministic), adjoint FP32 rel-l2 <= 1e-6.
"""
import numpy as np
import pytest
import torch

import nfftm

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(torch.linalg.vector_norm(a - b) / torch.linalg.vector_norm(b))


@pytest.mark.parametrize("change", ["nodes", "set_tiles"])
def test_change_waits_for_the_batch(change):
    print(f"batch in flight, {change}", flush=True)
    rng = np.random.default_rng(3)
    sizes = [((256, 256), 200000), ((160, 200), 150000)]
    ks = [rng.random((2, M)) - 0.5 for _, M in sizes]
    plans = [nfftm.plan_nfft(k, N, m=4, sigma=2.0, precompute=nfftm.LINEAR, dtype=torch.float32)
             for k, (N, _) in zip(ks, sizes)]
    b = nfftm.BatchPlan(plans, [4, 2], autotune=False)
    own = [i for i, _ in b.slots]
    fs = [torch.randn(plans[i].N, dtype=torch.complex64, device="cuda") for i in own]
    hs = [torch.randn((plans[i].J,), dtype=torch.complex64, device="cuda") for i in own]
    want, wantH = [y.clone() for y in b.forward(fs)], [x.clone() for x in b.adjoint(hs)]
    a = torch.randn((4096, 4096), device="cuda")
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        for _ in range(20):  # some ms before the batch
            a = (a @ a).clamp(-1, 1)
        got = [b.forward(fs) for _ in range(5)]
        gotH = [b.adjoint(hs) for _ in range(5)]
    if change == "nodes":
        for p, k in zip(plans, ks):
            p.nodes_(np.ascontiguousarray(0.3 * k[:, ::-1]))
    else:
        for p in plans:
            p.set_tiles(32, 256)
    torch.cuda.synchronize()
    for ys, xs in zip(got, gotH):
        for y, w in zip(ys, want):
            assert torch.equal(y, w)
        for x, w in zip(xs, wantH):
            assert rel(x, w) < 1e-6
    with pytest.raises(nfftm.ArgumentError):  # the batch is of the old nodes
        b.forward(fs)
