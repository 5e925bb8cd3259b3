"""Performance cases: what users of this library have it do on one GPU.

Each case is one pass of a program's time step through the public entry
points (``accfft_amd.Plan``, ``accfft_amd.autograd``) on device-resident
fields; plans and output buffers are made once, as a solver keeps them.

Keys of a case:
    op         forward    execute_r2c                      -> half spectrum
               roundtrip  execute_r2c, execute_c2r         -> N x the field
               c2c        execute_c2c forward              -> spectrum
               c2c_back   forward and backward c2c         -> N x the field
               laplace, inv_laplace, grad, divergence      -> real field(s)
               loss       0.5 ||div(grad(invlap u)) - g||^2 through
                          torch.autograd, forward and backward
               slab       execute_r2c of one rank's share of a P x 1 grid
                          (exchange = identity)
    n0 n1 n2   the grid (slab: the global grid), z fastest
    fp64       double precision
    ranks      slab: P

Plans are made with the default flag, ACCFFT_MEASURE, as bench.py does.
"""
import math

import torch

import accfft_amd as af
from accfft_amd import autograd as ag

MAX_POINTS = 512 ** 3


def _case(name, op, n, fp64, ranks=1):
    return {"name": name, "op": op, "n0": n[0], "n1": n[1], "n2": n[2], "fp64": fp64,
            "ranks": ranks}


def listed():
    return [
        # the plain method of the reference's first step: a small FP64 grid,
        # where launches and their latency count
        _case("roundtrip_64_f64", "roundtrip", (64, 64, 64), True),
        # odd and prime axes, as in the random-shape tests
        _case("roundtrip_61x45x70_f64", "roundtrip", (61, 45, 70), True),
        # a grid of mixed small factors (non-cubic box) with an odd z length
        _case("c2c_back_120x200x75_f32", "c2c_back", (120, 200, 75), False),
        # the usual production size, one direction
        _case("forward_256_f32", "forward", (256, 256, 256), False),
        # the headline: a spectral solver's transform pair
        _case("roundtrip_512_f32", "roundtrip", (512, 512, 512), False),
        # the same in the reference's default precision
        _case("roundtrip_512_f64", "roundtrip", (512, 512, 512), True),
        # complex fields (wave functions) at the headline size
        _case("c2c_512_f32", "c2c", (512, 512, 512), False),
        # turbulence / dealiased grids: 3/2 of a power of two
        _case("roundtrip_384_f32", "roundtrip", (384, 384, 384), False),
        # a large 3/2-rule grid in FP64
        _case("forward_768_f64", "forward", (768, 768, 768), True),
        # a spectral operator (diffusion step, Poisson-like solves)
        _case("laplace_512_f32", "laplace", (512, 512, 512), False),
        # the differentiable loss: gradient and divergence (per-axis
        # derivatives), inverse Laplacian and their adjoints
        _case("loss_256_f32", "loss", (256, 256, 256), False),
        # one rank's share of 2048^3 on 8 ranks
        _case("slab_2048_f32", "slab", (2048, 2048, 2048), False, 8),
    ]


def _smooth(rng, lo, hi):
    """A length whose prime factors are 2, 3, 5 and 7, spread over log(lo) ... log(hi)."""
    while True:
        v = round(math.exp(rng.uniform(math.log(lo), math.log(hi))))
        m = v
        for f in (2, 3, 5, 7):
            while m % f == 0:
                m //= f
        if m == 1:
            return v


def draw(rng):
    """Grids of 16 to 512 points an axis: powers of two, lengths with small
    factors (what FFT users pick when a power of two does not fit), and now
    and then any length at all."""
    op = rng.choice(["forward", "roundtrip", "roundtrip", "roundtrip", "c2c", "c2c_back",
                     "laplace", "inv_laplace", "grad", "divergence"])
    fp64 = rng.random() < 0.5
    kind = rng.random()
    while True:
        if kind < 0.25:
            n = [2 ** rng.randint(4, 9) for _ in range(3)]
        elif kind < 0.45:
            n = [_smooth(rng, 16, 512)] * 3
        elif kind < 0.85:
            n = [_smooth(rng, 16, 512) for _ in range(3)]
        else:
            n = [round(math.exp(rng.uniform(math.log(16), math.log(300)))) for _ in range(3)]
        if 4096 <= n[0] * n[1] * n[2] <= MAX_POINTS:
            break
    c = _case("", op, n, fp64)
    del c["name"]
    return c


def _n(case):
    return (case["n0"], case["n1"], case["n2"])


def _dtypes(case):
    return ((torch.float64, torch.complex128) if case["fp64"]
            else (torch.float32, torch.complex64))


def _inputs(case, seed):
    """The input fields: N(0, 1), on the plain method's grid sin x + sin y +
    sin z plus small noise; the loss takes a second, smooth field g."""
    real, cplx = _dtypes(case)
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed))
    n = _n(case)
    op = case["op"]
    if op == "slab":
        return [torch.randn((n[0] // case["ranks"], n[1], n[2]), generator=g, device=dev,
                            dtype=real)]
    if op in ("c2c", "c2c_back"):
        return [torch.view_as_complex(torch.randn(n + (2,), generator=g, device=dev, dtype=real))]
    if op == "divergence":
        return [torch.randn(n, generator=g, device=dev, dtype=real) for _ in range(3)]
    x = torch.randn(n, generator=g, device=dev, dtype=real)
    if n == (64, 64, 64):
        t = torch.sin(2 * math.pi * torch.arange(64, device=dev, dtype=real) / 64)
        x = t[:, None, None] + t[None, :, None] + t[None, None, :] + 1e-3 * x
    if op != "loss":
        return [x]
    # the target: a sum of plane waves of falling amplitude
    w = torch.zeros(n, device=dev, dtype=real)
    ax = [2 * math.pi * torch.arange(m, device=dev, dtype=real) / m for m in n]
    k = torch.randint(1, 9, (6, 3), generator=g, device=dev).tolist()
    for a, b, c in k:
        ph = a * ax[0][:, None, None] + b * ax[1][None, :, None] + c * ax[2][None, None, :]
        w += torch.cos(ph) / float(a * a + b * b + c * c)
    return [x, w]


def prepare(case, seed):
    real, cplx = _dtypes(case)
    prec = af.F64 if case["fp64"] else af.F32
    n, op = _n(case), case["op"]
    x = _inputs(case, seed)
    dev = x[0].device
    half = (n[0], n[1], n[2] // 2 + 1)
    s = {"op": op, "x": x}
    if op == "loss":
        s["S"] = ag.Spectral(n, real, dev)
        s["u"] = x[0].requires_grad_(True)
    elif op == "slab":
        P = case["ranks"]
        s["spec"] = torch.empty((n[0], n[1] // P, half[2]), dtype=cplx, device=dev)
        s["plan"] = af.Plan("r2c_slab", n, x[0], s["spec"], prec, nprocs=P)
    elif op in ("c2c", "c2c_back"):
        s["spec"] = torch.empty(n, dtype=cplx, device=dev)
        s["plan"] = af.Plan("c2c", n, x[0], s["spec"], prec)
        if op == "c2c_back":
            s["back"] = torch.empty_like(x[0])
    elif op in ("forward", "roundtrip"):
        s["spec"] = torch.empty(half, dtype=cplx, device=dev)
        s["plan"] = af.Plan("r2c", n, x[0], s["spec"], prec)
        if op == "roundtrip":
            s["back"] = torch.empty_like(x[0])
    else:
        s["out"] = [torch.empty_like(x[0]) for _ in range(3 if op == "grad" else 1)]
        s["plan"] = af.Plan("r2c", n, x[0], s["out"][0], prec)
    return s


def run(s):
    op, x = s["op"], s["x"]
    if op == "loss":
        u, S = s["u"], s["S"]
        u.grad = None
        v = ag.divergence(*ag.grad(ag.inv_laplace(u, S), S), S)
        loss = 0.5 * torch.sum((v - x[1]) ** 2)
        loss.backward()
        return {"loss": loss.detach(), "grad": u.grad}
    p = s["plan"]
    if op in ("forward", "slab"):
        p.execute_r2c(x[0], s["spec"])
        return s["spec"]
    if op == "roundtrip":
        p.execute_r2c(x[0], s["spec"])
        p.execute_c2r(s["spec"], s["back"])
        return s["back"]
    if op == "c2c":
        p.execute_c2c(af.ACCFFT_FORWARD, x[0], s["spec"])
        return s["spec"]
    if op == "c2c_back":
        p.execute_c2c(af.ACCFFT_FORWARD, x[0], s["spec"])
        p.execute_c2c(af.ACCFFT_BACKWARD, s["spec"], s["back"])
        return s["back"]
    if op == "grad":
        p.grad(x[0], *s["out"])
        return s["out"]
    if op == "divergence":
        p.divergence(*x, s["out"][0])
    else:
        getattr(p, op)(x[0], s["out"][0])
    return s["out"][0]


def work(case):
    """Each field read once and written once (a transform pair writes the
    spectrum and reads it again: it is the program's own array)."""
    n, op = _n(case), case["op"]
    N = float(n[0]) * n[1] * n[2]
    s = 8.0 if case["fp64"] else 4.0
    R, C, Z = N * s, float(n[0]) * n[1] * (n[2] // 2 + 1) * 2 * s, 2 * N * s
    fft = 2.5 * N * math.log2(N)  # one real 3-D transform
    P = case["ranks"]
    return {
        "forward": lambda: {"bytes": R + C, "flops": fft},
        "roundtrip": lambda: {"bytes": 2 * (R + C), "flops": 2 * fft},
        "c2c": lambda: {"bytes": 2 * Z, "flops": 2 * fft},
        "c2c_back": lambda: {"bytes": 4 * Z, "flops": 4 * fft},
        "laplace": lambda: {"bytes": 2 * R, "flops": 2 * fft},
        "inv_laplace": lambda: {"bytes": 2 * R, "flops": 2 * fft},
        # one 1-D transform pair per component
        "grad": lambda: {"bytes": 4 * R, "flops": 2 * fft},
        "divergence": lambda: {"bytes": 4 * R, "flops": 2 * fft},
        # inverse Laplacian, gradient, divergence, and back: u, g read, the
        # gradient written
        "loss": lambda: {"bytes": 3 * R, "flops": 12 * fft},
        "slab": lambda: {"bytes": (R + C) / P, "flops": fft / P},
    }[op]()


def _wave(m, dtype=torch.float64):
    """Signed wavenumbers 0 ... m-1 with the entry at m/2 (integer division)
    zero, as the reference's multipliers have them."""
    k = torch.arange(m, dtype=dtype)
    w = torch.where(k > m // 2, k - m, k)
    w[m // 2] = 0
    return w


def _deriv(x, d):
    """The per-axis spectral derivative i w(k): the modes at m/2 (integer
    division) and their mirror images are zero."""
    m = x.shape[d]
    w = _wave(m)
    w[(m - m // 2) % m] = 0
    shape = [1, 1, 1]
    shape[d] = m
    return torch.fft.ifft(torch.fft.fft(x, dim=d) * (1j * w.reshape(shape)), dim=d).real


def _symbol(n):
    nh = n[2] // 2 + 1
    w = [_wave(n[0])[:, None, None], _wave(n[1])[None, :, None], _wave(n[2])[None, None, :nh]]
    return -(w[0] ** 2 + w[1] ** 2 + w[2] ** 2)


def exact(case, seed):
    n, op = _n(case), case["op"]
    N = float(n[0]) * n[1] * n[2]
    x = [v.cpu().to(torch.complex128 if v.is_complex() else torch.float64)
         for v in _inputs(case, seed)]
    if op == "forward":
        return torch.fft.rfftn(x[0])
    if op == "roundtrip":
        return torch.fft.irfftn(torch.fft.rfftn(x[0]), s=n) * N
    if op == "c2c":
        return torch.fft.fftn(x[0])
    if op == "c2c_back":
        return torch.fft.ifftn(torch.fft.fftn(x[0])) * N
    if op in ("laplace", "inv_laplace"):
        f = _symbol(n)
        if op == "inv_laplace":
            f = torch.where(f == 0, torch.zeros_like(f), 1.0 / f)
        return torch.fft.irfftn(torch.fft.rfftn(x[0]) * f, s=n)
    if op == "grad":
        return [_deriv(x[0], d) for d in range(3)]
    if op == "divergence":
        return _deriv(x[0], 0) + _deriv(x[1], 1) + _deriv(x[2], 2)
    if op == "loss":
        u, g = x
        # div grad invlap is the projection onto the modes with a wavenumber
        keep = (_symbol(n) != 0).to(torch.float64)

        def project(v):
            return torch.fft.irfftn(torch.fft.rfftn(v) * keep, s=n)

        r = project(u) - g
        return {"loss": 0.5 * torch.sum(r * r), "grad": project(r)}
    # slab: z and y transforms of the share, the exchange blocks [P][n0][n1]
    # stacked along x (the identity exchange), the x transform
    P = case["ranks"]
    n0, n1 = n[0] // P, n[1] // P
    zy = torch.fft.rfftn(x[0], dim=(1, 2))
    got = zy.reshape(n0, P, n1, zy.shape[2]).transpose(0, 1).reshape(n[0], n1, zy.shape[2])
    return torch.fft.fft(got, dim=0)
