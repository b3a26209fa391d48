"""The workloads that the library's speed is measured on, each through the public transforms.

A case is a dict: ``kind`` (1, 2 or 3: the transform's type; "grad": a type 2 followed by a
type 1 with gradients), ``dim``, ``M`` points, ``n1 .. n_dim`` modes, ``eps``, ``batch``
(transforms that share the points), ``points`` (their distribution) and ``double`` (complex128
instead of complex64).  Type 3 has ``N`` targets in [-s_max, s_max]^dim instead of modes.
"""

from __future__ import annotations

import math

import torch

import nufftax_amd as N

PI = math.pi


def _case(name, kind, dim, M, modes, eps=1e-6, batch=1, points="uniform", double=False, **more):
    c = {"name": name, "kind": kind, "dim": dim, "M": M, "eps": eps, "batch": batch, "points": points,
         "double": double}
    c.update({f"n{d + 1}": n for d, n in enumerate(modes)})
    c.update(more)
    return {k: v for k, v in c.items() if not (k == "name" and v is None)}


def listed():
    return [
        # one short signal: a call whose time is launches and host work
        _case("1d-t1-1k", 1, 1, 1000, (64,)),
        # an irregularly sampled signal of ordinary length
        _case("1d-t1-100k", 1, 1, 100_000, (1024,)),
        # a long time series evaluated at irregular times; the grid (2 million cells) is no power of two
        _case("1d-t2-1M-modes", 2, 1, 3_000_017, (1_000_000,)),
        # an MRI slice from 8 receive coils that share one trajectory; ragged sizes
        _case("2d-t1-8-coils", 1, 2, 213_001, (200, 184), batch=8, points="radial"),
        # radial MRI gridding at full size, adjoint and forward operator
        _case("2d-t1-radial-4M", 1, 2, 3_999_744, (512, 512), points="radial"),
        _case("2d-t2-radial-4M", 2, 2, 3_999_744, (512, 512), points="radial"),
        # one step of a reconstruction that also fits its trajectory: forward and backward
        _case("2d-grad-1M", "grad", 2, 1_000_000, (256, 256)),
        # particles in clusters to Fourier modes and back, the largest calls
        _case("3d-t1-clusters-8M", 1, 3, 8_000_000, (128, 128, 128), points="clusters"),
        _case("3d-t2-clusters-8M", 2, 3, 8_000_000, (128, 128, 128), points="clusters"),
        # the same at low accuracy, on a grid that is no power of two
        _case("3d-t1-eps-1e-4", 1, 3, 1_500_000, (100, 96, 90), eps=1e-4),
        # high accuracy in double precision
        _case("3d-t1-complex128", 1, 3, 500_000, (64, 64, 64), eps=1e-12, points="clusters", double=True),
        # scattered sources to scattered frequencies (crystallography, boundary integrals)
        _case("3d-t3-complex128", 3, 3, 200_000, (), eps=1e-9, double=True, N=200_000, s_max=64.0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["1d", "1d", "2d", "2d", "2d", "grad", "3d", "3d", "3d double", "type 3"])
    kind = rng.choice([1, 2])
    if family == "1d":
        return _case(None, kind, 1, _log(rng, 1000, 3_000_000), (_log(rng, 64, 1_000_000),),
                     eps=rng.choice([1e-6, 1e-4]))
    if family == "2d":
        batch = rng.choice([1, 1, 1, 4, 8])
        return _case(None, kind, 2, _log(rng, 10_000, 4_000_000 // batch), tuple(_log(rng, 64, 512) for _ in range(2)),
                     eps=rng.choice([1e-6, 1e-6, 1e-4]), batch=batch, points=rng.choice(["uniform", "radial"]))
    if family == "grad":
        return _case(None, "grad", 2, _log(rng, 10_000, 1_000_000), tuple(_log(rng, 64, 256) for _ in range(2)),
                     points=rng.choice(["uniform", "radial"]))
    if family == "3d":
        return _case(None, kind, 3, _log(rng, 100_000, 8_000_000), tuple(_log(rng, 32, 128) for _ in range(3)),
                     eps=rng.choice([1e-6, 1e-6, 1e-4]), points=rng.choice(["uniform", "clusters"]))
    if family == "3d double":
        return _case(None, kind, 3, _log(rng, 50_000, 500_000), tuple(_log(rng, 32, 64) for _ in range(3)),
                     eps=rng.choice([1e-9, 1e-12]), points=rng.choice(["uniform", "clusters"]), double=True)
    return _case(None, 3, 3, _log(rng, 20_000, 200_000), (), eps=1e-9, double=True, N=_log(rng, 20_000, 200_000),
                 s_max=round(rng.uniform(16.0, 64.0), 3))


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _modes(case):
    return tuple(case[f"n{d + 1}"] for d in range(case["dim"]))


def _points(case, g, dev):
    dim, M = case["dim"], case["M"]
    rand = lambda *s: torch.rand(*s, generator=g, device=dev, dtype=torch.float64)  # noqa: E731
    randn = lambda *s: torch.randn(*s, generator=g, device=dev, dtype=torch.float64)  # noqa: E731
    wrap = lambda v: torch.remainder(v + PI, 2 * PI) - PI  # noqa: E731
    if case["points"] == "radial":  # spokes of random angle, radius uniform, jitter 1e-3
        spokes = max(16, min(512, M // 512))
        theta = rand(spokes) * PI
        theta = theta[torch.arange(M, device=dev) * spokes // M]
        r = (2 * rand(M) - 1) * PI
        return [wrap(r * torch.cos(theta) + 1e-3 * randn(M)), wrap(r * torch.sin(theta) + 1e-3 * randn(M))]
    if case["points"] == "clusters":  # 16 Gaussians of sigma 0.3
        centres = (2 * rand(16, dim) - 1) * PI
        label = torch.randint(16, (M,), generator=g, device=dev)
        return [wrap(centres[label, d] + 0.3 * randn(M)) for d in range(dim)]
    return [(2 * rand(M) - 1) * PI for _ in range(dim)]


def _inputs(case, seed):
    """coords, targets, source (strengths or modes), and the gradient case's image, as given to the call."""
    dev = _device()
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    rdt, cdt = (torch.float64, torch.complex128) if case["double"] else (torch.float32, torch.complex64)
    randn = lambda *s: torch.randn(*s, generator=g, device=dev, dtype=cdt) * math.sqrt(2.0)  # noqa: E731
    coords = [x.to(rdt) for x in _points(case, g, dev)]
    targets, image = [], None
    lead = (case["batch"],) if case["batch"] > 1 else ()
    if case["kind"] in (1, 3):
        source = randn(*lead, case["M"])
    else:
        source = randn(*lead, *reversed(_modes(case)))
    if case["kind"] == 3:
        targets = [((2 * torch.rand(case["N"], generator=g, device=dev, dtype=torch.float64) - 1) * case["s_max"]).to(rdt)
                   for _ in range(case["dim"])]
    if case["kind"] == "grad":
        image = randn(*reversed(_modes(case)))
    return coords, targets, source, image


def prepare(case, seed):
    coords, targets, source, image = _inputs(case, seed)
    state = {"kind": case["kind"], "dim": case["dim"], "eps": case["eps"], "coords": coords, "targets": targets,
             "source": source, "image": image}
    if case["kind"] == 3:  # the grid from the known extents of sources and targets
        state["modes"] = (N.compute_type3_grid_size(PI, case["s_max"], eps=case["eps"]),) * case["dim"]
    else:
        state["modes"] = _modes(case)
    if case["dim"] == 1:
        state["modes"] = state["modes"][0]
    return state


def run(state):
    kind, dim, eps, coords, source = (state[k] for k in ("kind", "dim", "eps", "coords", "source"))
    if kind == "grad":
        x, y, f = (v.detach().requires_grad_(True) for v in (*coords, source))
        out = N.nufft2d1(x, y, N.nufft2d2(x, y, f, eps=eps), state["modes"], eps=eps)
        loss = torch.sum(torch.abs(out - state["image"]) ** 2)
        return [out.detach(), *torch.autograd.grad(loss, (f, x, y))]
    if kind == 1:
        return getattr(N, f"nufft{dim}d1")(*coords, source, state["modes"], eps=eps)
    if kind == 2:
        return getattr(N, f"nufft{dim}d2")(*coords, source, eps=eps)
    return getattr(N, f"nufft{dim}d3")(*coords, source, *state["targets"], state["modes"], eps=eps)


def work(case):
    """Each input read once and each output written once; the products of the points with a
    kernel of the width that eps asks for, and the FFT of a grid of twice the modes."""
    dim, M, batch = case["dim"], case["M"], case["batch"]
    real, cplx = (8, 16) if case["double"] else (4, 8)
    width = math.ceil(-math.log10(case["eps"])) + 1
    spread = 4.0 * M * width**dim
    if case["kind"] == 3:
        n = case["N"]
        cells = (4.0 * case["s_max"] + width) ** dim * 2**dim
        return {"bytes": dim * real * (M + n) + cplx * (M + n),
                "flops": 4.0 * (M + n) * width**dim + 5 * cells * math.log2(cells)}
    modes = math.prod(_modes(case))
    cells = modes * 2**dim
    fft = 5 * cells * math.log2(cells)
    if case["kind"] == "grad":  # coordinates, modes and image in; image and gradients out; two forward and two adjoint passes
        return {"bytes": 2 * dim * real * M + 4 * cplx * modes, "flops": 4 * (spread + fft)}
    return {"bytes": dim * real * M + batch * cplx * (M + modes), "flops": batch * (spread + fft)}


# ---------------------------------------------------------------- the direct sums in 64 bits


def _factors(coords, modes, sign):
    """The two factors of exp(i sign k.x) for a chunk of points: left (A, m), right (B, m), every
    mode being one row of the outer product (1D: k = hi * B + lo; 2D: k2, k1; 3D: (k3, k2), k1)."""
    def e(k, x):
        return torch.polar(torch.ones((), dtype=torch.float64, device=x.device), sign * k[:, None] * x[None, :])

    def kv(n):
        return torch.arange(-(n // 2), (n + 1) // 2, device=coords[0].device, dtype=torch.float64)

    if len(modes) == 1:
        n = modes[0]
        b = math.isqrt(n - 1) + 1
        a = -(-n // b)
        hi = torch.arange(a, device=coords[0].device, dtype=torch.float64) * b - n // 2
        return e(hi, coords[0]), e(torch.arange(b, device=coords[0].device, dtype=torch.float64), coords[0])
    right = e(kv(modes[0]), coords[0])
    left = e(kv(modes[1]), coords[1])
    if len(modes) == 3:
        left = (e(kv(modes[2]), coords[2])[:, None, :] * left[None, :, :]).reshape(-1, left.shape[-1])
    return left, right


def _chunks(M, modes):
    rows = modes[1] * (modes[2] if len(modes) == 3 else 1) if len(modes) > 1 else math.isqrt(modes[0]) + 1
    m = max(1024, min(65536, (1 << 26) // rows))
    return [(s, min(M, s + m)) for s in range(0, M, m)]


def _direct1(coords, c, modes, sign):
    """sum_j c[t, j] exp(i sign k.x_j), c (batch, M) -> (batch, n3, n2, n1)."""
    n = math.prod(modes)
    out = None
    for s, e in _chunks(c.shape[-1], modes):
        left, right = _factors([x[s:e] for x in coords], modes, sign)
        if out is None:
            out = [torch.zeros(left.shape[0], right.shape[0], dtype=torch.complex128, device=c.device) for _ in c]
        rt = right.T.contiguous()
        for t in range(c.shape[0]):
            out[t].addmm_(left * c[t, s:e], rt)
    return torch.stack([o.reshape(-1)[:n].reshape(tuple(reversed(modes))) for o in out])


def _direct2(coords, f, modes, sign):
    """sum_k f[t, k] exp(i sign k.x_j), f (batch, n3, n2, n1) -> (batch, M)."""
    n, M = math.prod(modes), coords[0].shape[0]
    out = torch.empty(f.shape[0], M, dtype=torch.complex128, device=f.device)
    for s, e in _chunks(M, modes):
        left, right = _factors([x[s:e] for x in coords], modes, sign)
        for t in range(f.shape[0]):
            F = torch.zeros(left.shape[0] * right.shape[0], dtype=torch.complex128, device=f.device)
            F[:n] = f[t].reshape(-1)
            out[t, s:e] = (left * (F.reshape(left.shape[0], right.shape[0]) @ right)).sum(0)
    return out


def _direct3(coords, c, targets, sign):
    X = torch.stack(coords, 1)  # (M, dim)
    cc = torch.stack([c.real, c.imag])  # (2, M)
    out = []
    step = max(256, (1 << 28) // X.shape[0])
    for s in range(0, targets[0].shape[0], step):
        ph = sign * (X @ torch.stack([t[s:s + step] for t in targets]))
        p, q = cc @ torch.cos(ph), cc @ torch.sin(ph)
        out.append(torch.complex(p[0] - q[1], p[1] + q[0]))
    return torch.cat(out)


def exact(case, seed):
    coords, targets, source, image = _inputs(case, seed)
    coords = [x.double() for x in coords]
    source = source.to(torch.complex128)
    if case["kind"] == 3:
        return _direct3(coords, source, [t.double() for t in targets], 1)
    modes = _modes(case)
    dim = len(modes)
    if case["kind"] == "grad":
        # o = T1(v), v = T2(f), loss = sum |o - g|^2; gradients as dL/dRe + i dL/dIm
        f = source[None]
        v = _direct2(coords, f, modes, -1)
        o = _direct1(coords, v, modes, 1)
        r = 2.0 * (o - image.to(torch.complex128))
        gv = _direct2(coords, r, modes, -1)
        gf = _direct1(coords, gv, modes, 1)
        gx = []
        for d in range(dim):
            k = torch.arange(-(modes[d] // 2), (modes[d] + 1) // 2, device=f.device, dtype=torch.float64)
            w = -1j * k.reshape([-1 if dim - 1 - a == d else 1 for a in range(dim)])
            dr, df = _direct2(coords, torch.cat([w * r, w * f]), modes, -1)
            gx.append((v[0] * dr.conj() + gv[0].conj() * df).real)
        return [o[0], gf[0], *gx]
    batched = source if case["batch"] > 1 else source[None]
    out = (_direct1(coords, batched, modes, 1) if case["kind"] == 1 else _direct2(coords, batched, modes, -1))
    return out if case["batch"] > 1 else out[0]
