"""Performance cases of the NFFT framework: the transforms that its users run.

Each case is a dict of plain values; `prepare` makes what a program holds
before the call (inputs on the GPU, plans), `run` is one pass through the
public entry points, `work` the bytes and operations that pass cannot do
without, `exact` the same outputs from plain torch in 64 bits (direct sums as
matrix products, or for long 1-D signals a 64-bit NUFFT with a 16-point
window).  `draw` gives further cases of the same ranges.

Kinds:
  transform  forward and adjoint of one plan (1-D signals, images, volumes)
  train      forward and both gradients through torch autograd (learned
             trajectories, trajectory correction)
  batch      many plans and shared-trajectory images in one BatchPlan
             (multi-coil, mixed trajectories)
  toeplitz   one normal-operator product of an iterative reconstruction
  sdc        sampling density compensation of a trajectory
  stack      a directional plan: stack-of-stars, every partition of a volume
             transformed along two axes
  renode     nodes! and a forward transform: a trajectory that moves from
             call to call
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.join(os.getcwd(), "nfft.jl_amd"))

import nfftm  # noqa: E402
from nfftm import autograd, tools  # noqa: E402

PRE = {"linear": nfftm.LINEAR, "polynomial": nfftm.POLYNOMIAL, "tensor": nfftm.TENSOR}
GOLDEN = math.pi * 2.0 / (1.0 + math.sqrt(5.0))


def listed():
    return [
        # a small image with few samples: latency and launches
        {"name": "image_64_f64", "kind": "transform", "N0": 64, "N1": 64, "N2": 0, "M": 4096, "nodes": "uniform",
         "dtype": "f64", "m": 4, "sigma": 2.0, "pre": "linear"},
        # one slice of a radial MRI scan with the plan's default parameters (reltol 1e-9: m = 5, sigma = 2)
        {"name": "radial_320_f64", "kind": "transform", "N0": 320, "N1": 320, "N2": 0, "M": 503 * 640,
         "nodes": "radial", "dtype": "f64", "m": 5, "sigma": 2.0, "pre": "polynomial"},
        # one training step of a learned spiral trajectory
        {"name": "spiral_train_256_f32", "kind": "train", "N0": 256, "N1": 256, "N2": 0, "M": 65536,
         "nodes": "spiral", "dtype": "f32", "m": 4, "sigma": 2.0, "pre": "polynomial"},
        # the headline volume: forward and adjoint of a 128^3 image
        {"name": "volume_128_f32", "kind": "transform", "N0": 128, "N1": 128, "N2": 128, "M": 2 ** 21,
         "nodes": "uniform", "dtype": "f32", "m": 4, "sigma": 2.0, "pre": "linear"},
        # a volume in double precision, default parameters
        {"name": "volume_96_f64", "kind": "transform", "N0": 96, "N1": 96, "N2": 96, "M": 10 ** 6,
         "nodes": "uniform", "dtype": "f64", "m": 5, "sigma": 2.0, "pre": "polynomial"},
        # 3-D radial ("kooshball") sampling of an anisotropic volume at moderate accuracy (reltol 1e-5: m = 3)
        {"name": "koosh_150x144x125_f32", "kind": "transform", "N0": 150, "N1": 144, "N2": 125, "M": 3001 * 300,
         "nodes": "radial", "dtype": "f32", "m": 3, "sigma": 2.0, "pre": "polynomial"},
        # a long signal, samples clustered at the ends, small oversampling: the largest call
        {"name": "signal_2p24_f32", "kind": "transform", "N0": 2 ** 24, "N1": 0, "N2": 0, "M": 2 ** 24,
         "nodes": "edges", "dtype": "f32", "m": 6, "sigma": 1.25, "pre": "tensor"},
        # mixed trajectories and a multi-coil radial image in one batch
        {"name": "batch_16x2d_8coils_f32", "kind": "batch", "N0": 256, "N1": 256, "N2": 0, "M": 402 * 512,
         "plans": 16, "coils": 8, "dtype": "f32", "m": 4, "sigma": 2.0, "pre": "linear"},
        # A'A of a 256^2 image through its Toeplitz kernel, as each iteration of a solver does
        {"name": "toeplitz_256_f32", "kind": "toeplitz", "N0": 256, "N1": 256, "N2": 0, "M": 402 * 512,
         "nodes": "radial", "dtype": "f32", "m": 4, "sigma": 2.0, "pre": "polynomial"},
        # density weights of a golden-angle radial trajectory, 20 iterations (the default)
        {"name": "sdc_radial_256_f32", "kind": "sdc", "N0": 256, "N1": 256, "N2": 0, "M": 402 * 512,
         "nodes": "radial", "dtype": "f32", "m": 4, "sigma": 2.0, "pre": "polynomial"},
        # stack-of-stars: 32 partitions of a 240^2 image on one radial trajectory
        {"name": "stack_32x240_f32", "kind": "stack", "N0": 32, "N1": 240, "N2": 240, "M": 256 * 480,
         "nodes": "radial", "dtype": "f32", "m": 4, "sigma": 2.0, "pre": "linear"},
        # a motion-corrected trajectory: new nodes from the host, then a forward transform
        {"name": "renode_256_f32", "kind": "renode", "N0": 256, "N1": 256, "N2": 0, "M": 402 * 512,
         "nodes": "radial", "dtype": "f32", "m": 4, "sigma": 2.0, "pre": "linear"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _edge(rng, lo, hi):
    """An image edge: half of them multiples of 8 or 10 (usual matrix sizes), the rest any number."""
    n = _log(rng, lo, hi)
    q = rng.choice([1, 1, 8, 10])
    return max(lo, n // q * q)


def draw(rng):
    kind = rng.choice(["transform", "transform", "transform", "transform", "train", "batch", "toeplitz", "sdc",
                       "stack", "renode"])
    c = {"kind": kind, "dtype": rng.choice(["f32", "f32", "f64"])}
    m, sigma = rng.choice([(3, 2.0), (4, 2.0), (4, 2.0), (5, 2.0), (6, 1.5)])
    c.update(m=m, sigma=sigma, pre=rng.choice(["linear", "polynomial", "polynomial", "tensor"]))
    if kind == "transform":
        D = rng.choice([1, 2, 2, 3, 3])
        if D == 1:
            N, nodes = (_log(rng, 500, 2 ** 22), 0, 0), rng.choice(["uniform", "edges"])
        elif D == 2:
            N, nodes = (_edge(rng, 48, 640), _edge(rng, 48, 640), 0), rng.choice(["uniform", "radial", "spiral"])
        else:
            N = tuple(_edge(rng, 32, 144) for _ in range(3))
            nodes = rng.choice(["uniform", "radial"])
        P = math.prod(n for n in N if n)
        # between a quarter of the image's pixels (undersampled) and twice as many
        c.update(N0=N[0], N1=N[1], N2=N[2], nodes=nodes, M=max(500, min(2 ** 22, int(P * math.exp(rng.uniform(-1.4, 0.7))))))
    elif kind == "batch":
        n = _edge(rng, 64, 320)
        c.update(N0=n, N1=n, N2=0, plans=rng.randint(3, 20), coils=rng.randint(1, 10), M=n * _log(rng, n // 2, 2 * n))
    elif kind == "stack":
        n = _edge(rng, 96, 320)
        c.update(N0=_log(rng, 4, 48), N1=n, N2=n, nodes="radial", M=2 * n * _log(rng, n // 4, n))
    else:
        n0, n1 = _edge(rng, 64, 384), _edge(rng, 64, 384)
        nodes = "spiral" if kind == "train" else "radial"
        c.update(N0=n0, N1=n1, N2=0, nodes=nodes, M=2 * n0 * _log(rng, n1 // 4, n1))
        if kind in ("train", "renode"):
            c["m"], c["sigma"] = rng.choice([(3, 2.0), (4, 2.0), (5, 2.0)])
        if kind in ("toeplitz", "sdc"):
            c["sigma"], c["m"] = 2.0, rng.choice([3, 4])
    # no more work than the headline volume (64-bit operations counted twice)
    limit = work(listed()[3])["flops"]
    while work(c)["flops"] * (2 if c["dtype"] == "f64" else 1) > limit:
        c["M"] //= 2
        if kind in ("batch", "stack"):
            n = "plans" if kind == "batch" else "N0"
            c[n] = max(1, c[n] // 2)
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _shape(case):
    return tuple(n for n in (case["N0"], case["N1"], case["N2"]) if n)


def _complex(case):
    return torch.complex128 if case["dtype"] == "f64" else torch.complex64


def _real(case):
    return torch.float64 if case["dtype"] == "f64" else torch.float32


def _device():
    return torch.device("cuda") if torch.cuda.is_available() else torch.device("cpu")


def _data(shape, dtype, seed, which):
    """N(0,1) real and imaginary parts, drawn in 64 bits and rounded to dtype."""
    dev = _device()
    g = torch.Generator(device=dev)
    g.manual_seed(1000 * int(seed) + which)
    return torch.randn(shape, dtype=torch.complex128, device=dev, generator=g).mul_(math.sqrt(2.0)).to(dtype)


def _nodes(kind, D, M, seed, which=0):
    """(D, M) float64 nodes in [-1/2, 1/2); the seed moves every one of them."""
    rng = np.random.default_rng([int(seed), which])
    if kind == "uniform":
        return rng.random((D, M)) - 0.5
    if kind == "edges":  # Beta(1/2, 1/2) - 1/2
        return (np.sin(0.5 * np.pi * rng.random((D, M))) ** 2 - 0.5) * (1.0 - 2.0 ** -40)
    if kind == "spiral":  # 8 interleaved Archimedean spirals
        q = np.arange(M) % 8
        t = (np.arange(M) // 8 + rng.random(M)) / (M // 8 + 1)
        th = 2 * np.pi * (16 * t + q / 8) + rng.random()
        return 0.5 * t * np.stack([np.cos(th), np.sin(th)])
    # radial: golden-angle spokes (2-D) or directions spread over the sphere (3-D)
    samples = max(8, int(round(math.sqrt(M)))) if D == 2 else max(8, int(round(M ** (1 / 3) * 3)))
    spokes = -(-M // samples)
    r = (np.arange(samples) + rng.random()) / samples - 0.5
    th = np.arange(spokes) * GOLDEN + rng.random() * np.pi
    if D == 2:
        u = np.stack([np.cos(th), np.sin(th)])
    else:
        z = (2 * np.arange(spokes) + 1) / spokes - 1
        s = np.sqrt(1 - z * z)
        u = np.stack([s * np.cos(2 * th), s * np.sin(2 * th), z])
    return np.ascontiguousarray((u[:, :, None] * r).reshape(D, -1)[:, :M])


def _params(case):
    return dict(m=case["m"], sigma=case["sigma"], precompute=PRE[case["pre"]], dtype=_real(case))


def _batch_specs(case, seed):
    """(N, k) of the batch's plans: uneven images on uniform nodes, then the shared radial trajectory."""
    shape = np.random.default_rng([case["plans"], case["N0"]])  # sizes belong to the case, not to the seed
    specs = []
    for q in range(case["plans"]):
        n = int(shape.choice([64, 96, 128, 200, 256]))
        M = int(round(10 ** shape.uniform(4, 5.5)))
        specs.append(((n, n), _nodes("uniform", 2, M, seed, 10 + q)))
    specs.append(((case["N0"], case["N1"]), _nodes("radial", 2, case["M"], seed)))
    return specs


def prepare(case, seed):
    kind, N, cd = case["kind"], _shape(case), _complex(case)
    M = case["M"]
    if kind == "transform":
        k = _nodes(case["nodes"], len(N), M, seed)
        return {"kind": kind, "plan": nfftm.plan_nfft(k, N, **_params(case)), "f": _data(N, cd, seed, 1),
                "fh": _data((M,), cd, seed, 2)}
    if kind == "train":
        k = _nodes(case["nodes"], 2, M, seed)
        kt = torch.as_tensor(k, device=_device()).requires_grad_(True)
        x = _data(N, cd, seed, 1).requires_grad_(True)
        return {"kind": kind, "plan": nfftm.plan_nfft(k, N, **_params(case)), "k": kt, "x": x,
                "ybar": _data((M,), cd, seed, 2)}
    if kind == "batch":
        plans = [nfftm.plan_nfft(k, n, **_params(case)) for n, k in _batch_specs(case, seed)]
        b = nfftm.BatchPlan(plans, [1] * case["plans"] + [case["coils"]])
        fs = [_data(plans[i].N, cd, seed, 100 + s) for s, (i, _) in enumerate(b.slots)]
        fh = [_data((plans[i].J,), cd, seed, 300 + s) for s, (i, _) in enumerate(b.slots)]
        return {"kind": kind, "plans": plans, "batch": b, "f": fs, "fh": fh}
    if kind == "toeplitz":
        k = _nodes(case["nodes"], 2, M, seed)
        lam = tools.calculateToeplitzKernel(N, k, m=case["m"], sigma=case["sigma"], dtype=cd)
        return {"kind": kind, "lam": lam, "top": tools.Toeplitz(N, cd), "x": _data(N, cd, seed, 1)}
    if kind == "sdc":
        k = _nodes(case["nodes"], 2, M, seed)
        return {"kind": kind, "plan": nfftm.plan_nfft(k, N, **_params(case))}
    if kind == "stack":
        k = _nodes(case["nodes"], 2, M, seed)
        return {"kind": kind, "plan": nfftm.plan_nfft(k, N, dims=range(1, 3), **_params(case)),
                "f": _data(N, cd, seed, 1), "fh": _data((N[0], M), cd, seed, 2)}
    if kind == "renode":
        k = _nodes(case["nodes"], 2, M, seed)
        return {"kind": kind, "plan": nfftm.plan_nfft(_nodes(case["nodes"], 2, M, seed, 1), N, **_params(case)),
                "k": k, "f": _data(N, cd, seed, 1)}
    raise ValueError(kind)


def run(state):
    kind = state["kind"]
    if kind in ("transform", "stack"):
        p = state["plan"]
        return {"fhat": p * state["f"], "f": p.H * state["fh"]}
    if kind == "train":
        y = autograd.nfft(state["k"], state["x"], plan=state["plan"])
        kbar, xbar = torch.autograd.grad(y, (state["k"], state["x"]), state["ybar"])
        return {"y": y, "kbar": kbar, "xbar": xbar}
    if kind == "batch":
        return {"fhat": state["batch"].forward(state["f"]), "f": state["batch"].adjoint(state["fh"])}
    if kind == "toeplitz":
        return tools.convolveToeplitzKernel_(state["x"].clone(), state["lam"], state["top"])
    if kind == "sdc":
        return tools.sdc(state["plan"])
    if kind == "renode":
        return state["plan"].nodes_(state["k"]) * state["f"]
    raise ValueError(kind)


# ---------------------------------------------------------------------------
# what one pass cannot do without
# ---------------------------------------------------------------------------
def _one_direction(N, Q, M, sc, m, slices=1):
    """One direction of one plan: nodes, image and node values once, the taps and the FFT of the oversampled grid."""
    D, P = len(N), math.prod(N)
    return (8 * D * M + slices * sc * (P + M),
            slices * (4 * M * (2 * m) ** D + 5 * Q * math.log2(Q)))


def _grid(N, sigma):
    return math.prod(int(math.ceil(sigma * n)) // 2 * 2 for n in N)


def work(case):
    kind, N, M, m = case["kind"], _shape(case), case["M"], case["m"]
    sc = 16 if case["dtype"] == "f64" else 8
    if kind == "stack":
        b, f = _one_direction(N[1:], _grid(N[1:], case["sigma"]), M, sc, m, N[0])
        return {"bytes": 2 * b, "flops": 2 * f}
    Q = _grid(N, case["sigma"])
    b, f = _one_direction(N, Q, M, sc, m)
    if kind == "transform":
        return {"bytes": 2 * b, "flops": 2 * f}
    if kind == "train":  # forward, adjoint, and the gradient's taps for each dimension
        return {"bytes": 2 * b + M * (sc + 16), "flops": 2 * f + 2 * 4 * M * (2 * m) ** 2}
    if kind == "batch":
        tb = tf = 0
        for n, k in _batch_specs(case, 0):
            s = case["coils"] if (n == N and k.shape[1] == M) else 1
            x, y = _one_direction(n, _grid(n, case["sigma"]), k.shape[1], sc, m, s)
            tb, tf = tb + 2 * x, tf + 2 * y
        return {"bytes": tb, "flops": tf}
    if kind == "toeplitz":  # x, lambda and the result; two FFTs of size 2N
        P = math.prod(N)
        return {"bytes": sc * (2 * P + 4 * P), "flops": 2 * 5 * 4 * P * math.log2(4 * P)}
    if kind == "sdc":  # nodes and weights; 20 spreadings and interpolations, then a forward and an adjoint
        return {"bytes": 16 * M + sc // 2 * M, "flops": 20 * 2 * 2 * M * (2 * m) ** 2 + 2 * f}
    return {"bytes": b + 16 * M, "flops": f}  # renode: the nodes from the host as well


# ---------------------------------------------------------------------------
# 64-bit values without this repository's code
# ---------------------------------------------------------------------------
def _phases(k, n):
    """exp(-2 pi i k (j - n // 2)), j < n, for a vector of nodes: (len(k), n)."""
    t = k[:, None] * torch.arange(-(n // 2), n - n // 2, dtype=torch.float64, device=k.device)
    t = (t - torch.round(t)) * (-2 * math.pi)
    return torch.complex(torch.cos(t), torch.sin(t))


def _chunk(N):
    return max(256, min(1 << 16, (1 << 28) // max(1, math.prod(N[:-1]) * 4)))


def _ndft(k, f):
    """sum_n f[n] exp(-2 pi i k_j . n) for every node."""
    N, D = f.shape, f.dim()
    out = []
    for c in torch.split(k, _chunk(N), dim=1):
        E = [_phases(c[d], N[d]) for d in range(D)]
        if D == 1:
            y = E[0] @ f
        else:
            y = (E[-1] @ f.reshape(-1, N[-1]).T.contiguous()).reshape(-1, *N[:-1])
            for d in range(D - 2, -1, -1):
                y = (y * E[d].reshape(len(y), *([1] * d), N[d])).sum(-1)
        out.append(y)
    return torch.cat(out)


def _ndft_adjoint(k, fh, N):
    """sum_j fh_j exp(+2 pi i k_j . n) on the image of size N."""
    D, n = len(N), _chunk(N)
    f = torch.zeros((math.prod(N[:-1]), N[-1]), dtype=torch.complex128, device=k.device)
    for c, v in zip(torch.split(k, n, dim=1), torch.split(fh, n)):
        E = [_phases(c[d], N[d]).conj().resolve_conj() for d in range(D)]
        a = v[:, None]
        for d in range(D - 1):
            a = (a[:, :, None] * E[d][:, None, :]).reshape(len(v), -1)
        f += a.T.contiguous() @ E[-1]
    return f.reshape(N)


_TAPS, _SHAPE = 16, math.pi * 16 * 0.75  # Kaiser-Bessel, 16 points at oversampling 2: about 1e-14


def _kb(u):
    """Window exp(-b) I0(b sqrt(1 - (2 u / w)^2))."""
    z = _SHAPE * torch.sqrt(torch.clamp(1 - (2 * u / _TAPS) ** 2, min=0))
    return torch.special.i0e(z) * torch.exp(z - _SHAPE)


def _kb_hat(n, G):
    """Its Fourier transform at frequency index n of a grid of G points."""
    q = torch.sqrt(_SHAPE ** 2 - (math.pi * _TAPS * n / G) ** 2)
    return _TAPS * 0.5 * (torch.exp(q - _SHAPE) - torch.exp(-q - _SHAPE)) / q


def _long(k, N, f=None, fh=None):
    """1-D transform (f) or adjoint (fh) through a 64-bit NUFFT with oversampling 2."""
    G = 2 * N
    n = torch.arange(-(N // 2), N - N // 2, device=k.device)
    x = (k % 1.0) * G
    c = torch.floor(x)
    scale = 1.0 / _kb_hat(n.double(), G)
    if f is not None:
        g = torch.zeros(G, dtype=torch.complex128, device=k.device)
        g[n % G] = f * scale
        g = torch.view_as_real(torch.fft.fft(g))
        y = torch.zeros((len(k), 2), dtype=torch.float64, device=k.device)
        for t in range(1 - _TAPS // 2, _TAPS // 2 + 1):
            y += _kb(x - c - t)[:, None] * g[((c + t) % G).long()]
        return torch.view_as_complex(y)
    g = torch.zeros((G, 2), dtype=torch.float64, device=k.device)
    v = torch.view_as_real(fh)
    for t in range(1 - _TAPS // 2, _TAPS // 2 + 1):
        g.index_add_(0, ((c + t) % G).long(), _kb(x - c - t)[:, None] * v)
    return (torch.fft.ifft(torch.view_as_complex(g)) * G)[n % G] * scale


def _kb_plan(u, m, sigma):
    """The plan's own Kaiser-Bessel window at u grid units."""
    b = math.pi * (2 - 1 / sigma)
    q = torch.sqrt(torch.clamp(m * m - u * u, min=1e-300))
    return torch.where(u.abs() < m, torch.sinh(b * q) / (q * math.pi), torch.zeros_like(u))


def _density(case, k, N):
    """Pipe & Menon weights: 20 iterations w <- w / (C C' w) with the first grid maximum divided out, then the least-squares scale."""
    m, dev = case["m"], k.device
    G = [int(math.ceil(case["sigma"] * n)) // 2 * 2 for n in N]
    taps = range(1 - m, m + 1)
    idx, wt = [], []
    for d in range(2):
        x = (k[d] % 1.0) * G[d]
        c = torch.floor(x)
        idx.append([((c + t) % G[d]).long() for t in taps])
        wt.append([_kb_plan(x - c - t, m, G[d] / N[d]) for t in taps])
    pairs = [(idx[0][a] * G[1] + idx[1][b], wt[0][a] * wt[1][b]) for a in range(2 * m) for b in range(2 * m)]
    w = torch.ones(k.shape[1], dtype=torch.float64, device=dev)
    top = None
    for _ in range(20):
        g = torch.zeros(G[0] * G[1], dtype=torch.float64, device=dev)
        for i, v in pairs:
            g.index_add_(0, i, v * w)
        top = g.max() if top is None else top
        g /= top
        t = torch.zeros_like(w)
        for i, v in pairs:
            t += v * g[i]
        w = w / (t / top)
    u = _ndft(k, torch.ones(N, dtype=torch.complex128, device=dev))
    v = _ndft_adjoint(k, u * w, N)
    return w * (v.real.sum() / (v.abs() ** 2).sum())


def exact(case, seed):
    kind, N, cd, M = case["kind"], _shape(case), _complex(case), case["M"]
    dev, wide = _device(), torch.complex128
    if kind == "batch":
        specs = _batch_specs(case, seed)
        slots = list(range(case["plans"])) + [case["plans"]] * case["coils"]
        ks = [torch.as_tensor(k, device=dev) for _, k in specs]
        fh, f = [], []
        for s, i in enumerate(slots):
            n, k = specs[i]
            fh.append(_ndft(ks[i], _data(n, cd, seed, 100 + s).to(wide)))
            f.append(_ndft_adjoint(ks[i], _data((k.shape[1],), cd, seed, 300 + s).to(wide), n))
        return {"fhat": fh, "f": f}
    k = torch.as_tensor(_nodes(case["nodes"], 2 if kind == "stack" else len(N), M, seed), device=dev)
    if kind == "stack":
        f, fh = _data(N, cd, seed, 1).to(wide), _data((N[0], M), cd, seed, 2).to(wide)
        return {"fhat": torch.stack([_ndft(k, x) for x in f]),
                "f": torch.stack([_ndft_adjoint(k, x, N[1:]) for x in fh])}
    if kind == "transform":
        f, fh = _data(N, cd, seed, 1).to(wide), _data((M,), cd, seed, 2).to(wide)
        if len(N) == 1 and N[0] * M > 1 << 28:
            return {"fhat": _long(k[0], N[0], f=f), "f": _long(k[0], N[0], fh=fh)}
        return {"fhat": _ndft(k, f), "f": _ndft_adjoint(k, fh, N)}
    if kind == "train":
        x, ybar = _data(N, cd, seed, 1).to(wide), _data((M,), cd, seed, 2).to(wide)
        kbar = []
        for d in range(2):
            n = torch.arange(-(N[d] // 2), N[d] - N[d] // 2, dtype=torch.float64, device=dev)
            dy = _ndft(k, x * n.reshape(-1, 1) if d == 0 else x * n) * (-2j * math.pi)
            kbar.append((ybar.conj() * dy).real)
        return {"y": _ndft(k, x), "kbar": torch.stack(kbar), "xbar": _ndft_adjoint(k, ybar, N)}
    if kind == "toeplitz":
        return _ndft_adjoint(k, _ndft(k, _data(N, cd, seed, 1).to(wide)), N)
    if kind == "sdc":
        return _density(case, k, N)
    return _ndft(k, _data(N, cd, seed, 1).to(wide))  # renode
