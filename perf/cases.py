"""The work a program has this package do, as measurable cases.

Four kinds, each through the package's public entry points:

* ``evolve1d`` / ``evolve2d``: split-operator evolution (Evolver1D / Evolver2D,
  one grid by itself or many grids advanced together);
* ``fft``: the FourierTransform plan, forward and inverse;
* ``born``: Born-series scattering (QuPerturbation2D / QuPerturbation3D) and
  the forward cross section of its result.

``listed()`` holds one case of each use, ``draw()`` more of the same ranges.
"""
import ctypes
import math

import numpy as np
import torch

from qusim_amd import _native as N
from qusim_amd.api import (BoundaryCondition, Evolver1D, Evolver2D, Options, QuPerturbation2D,
                           QuPerturbation3D, SolverMethod, advance_batched)
from qusim_amd.fft import FourierTransform

_O4_T = 2.0 ** (1.0 / 3.0)


def listed():
    return [
        # the smallest call: one step of a short line, then its norm, as an
        # interactive program prints it after every step
        dict(name="evolve1d_256_step_norm", kind="evolve1d", n=256, precision="fp64", order=2,
             wall=False, count=1, steps=1, norm=True),
        # tunnelling probability against the grid size: lines of 1000 to 4000
        # points, fourth order
        dict(name="evolve1d_1000_o4", kind="evolve1d", n=1000, precision="fp64", order=4,
             wall=False, count=1, steps=20, norm=False),
        # the infinite-wall boundary (sine transform)
        dict(name="evolve1d_wall_1500", kind="evolve1d", n=1500, precision="fp64", order=2,
             wall=True, count=1, steps=20, norm=False),
        # a request loop's lane of 1D packets advanced together
        dict(name="evolve1d_32x4096_mixed32", kind="evolve1d", n=4096, precision="mixed32",
             order=2, wall=False, count=32, steps=50, norm=False),
        # the headline grid: 1024^2 in complex128 with an absorbing layer
        dict(name="evolve2d_1024_fp64", kind="evolve2d", nx=1024, ny=1024, precision="fp64",
             order=2, absorb=True, count=1, steps=20),
        # a grid chosen by the box and the spacing, not by the transform
        dict(name="evolve2d_750x600_o4", kind="evolve2d", nx=750, ny=600, precision="fp64",
             order=4, absorb=False, count=1, steps=5),
        # a request loop's lane of 2D packets in the mixed form
        dict(name="evolve2d_8x512_mixed32", kind="evolve2d", nx=512, ny=512,
             precision="mixed32", order=2, absorb=True, count=8, steps=20),
        # a grid that streams from HBM
        dict(name="evolve2d_4096_fp64", kind="evolve2d", nx=4096, ny=4096, precision="fp64",
             order=2, absorb=False, count=1, steps=4),
        # the transform plan by itself, there and back
        dict(name="fft3d_100x120x90", kind="fft", dims="100x120x90", precision=64),
        # a 2D scattering request
        dict(name="born2d_512_mixed32", kind="born", dims="512x512", precision="mixed32",
             energies=1, pre="Vellekoop", iters=40),
        # a 3D scattering solve in full precision on a grid of 96 points a side
        dict(name="born3d_96_fp64", kind="born", dims="96x96x96", precision="fp64", energies=2,
             pre="Hao1", iters=6),
        # many energies on one 3D grid with complex64 iterates
        dict(name="born3d_128_16e_mixed32", kind="born", dims="128x128x128",
             precision="mixed32", energies=16, pre="Vellekoop", iters=20),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _length(rng, lo, hi):
    """A line length as programs choose them: a power of two, a round number
    or (one in four) whatever the box divided by the spacing gives."""
    n = max(lo, min(hi, _log_int(rng, lo, hi)))
    how = rng.randrange(4)
    if how == 0:
        p = 1 << (n.bit_length() - 1)
        return p if p >= lo else 2 * p
    if how in (1, 2):
        q = 50 if n >= 500 else 10 if n >= 100 else 4
        return max(lo, n // q * q)
    return n


def draw(rng):
    what = rng.randrange(7)
    if what == 0:
        wall = rng.random() < 0.3
        return dict(kind="evolve1d", n=_length(rng, 100, 2500 if wall else 5000),
                    precision="fp64", order=rng.choice([2, 2, 4]), wall=wall, count=1,
                    steps=rng.choice([1, 5, 20]), norm=rng.random() < 0.5)
    if what == 1:
        return dict(kind="evolve1d", n=1 << rng.randrange(10, 14), precision="mixed32", order=2,
                    wall=False, count=rng.randrange(2, 65), steps=rng.randrange(10, 81),
                    norm=False)
    if what == 2:
        return dict(kind="evolve2d", nx=_length(rng, 64, 1600), ny=_length(rng, 64, 1600),
                    precision="fp64", order=rng.choice([2, 2, 4]), absorb=rng.random() < 0.5,
                    count=1, steps=rng.randrange(1, 7))
    if what == 3:
        n = 1 << rng.randrange(8, 11)
        return dict(kind="evolve2d", nx=n, ny=n, precision="mixed32", order=2,
                    absorb=rng.random() < 0.5, count=rng.randrange(1, 9),
                    steps=rng.randrange(5, 21))
    if what == 4:
        rank = rng.randrange(1, 4)
        hi = {1: 5000, 2: 1500, 3: 160}[rank]
        dims = [_length(rng, 12, hi) for _ in range(rank)]
        prec = 64
        if rng.random() < 0.4:
            prec = 32
        return dict(kind="fft", dims="x".join(str(d) for d in dims), precision=prec)
    if what == 5:
        if rng.random() < 0.5:
            return dict(kind="born", dims="%dx%d" % ((1 << rng.randrange(8, 11),) * 2),
                        precision="mixed32", energies=1, pre="Vellekoop",
                        iters=rng.randrange(10, 61))
        return dict(kind="born", dims="%dx%d" % (_length(rng, 160, 800), _length(rng, 160, 800)),
                    precision="fp64", energies=1, pre=rng.choice(["Vellekoop", "Hao1", "Hao2"]),
                    iters=rng.randrange(4, 13))
    if rng.random() < 0.5:
        return dict(kind="born", dims="x".join(["%d" % (64 << rng.randrange(2))] * 3),
                    precision="mixed32", energies=rng.randrange(1, 17), pre="Vellekoop",
                    iters=rng.randrange(5, 21))
    return dict(kind="born", dims="x".join(str(_length(rng, 40, 128)) for _ in range(3)),
                precision="fp64", energies=rng.randrange(1, 4), pre=rng.choice(["Vellekoop", "Hao1"]),
                iters=rng.randrange(3, 9))


# ------------------------------------------------------------------ inputs
# Grid spacings and time steps as in the repository's workloads: 0.1 (1D) and
# 0.3 (2D) with packets of momentum about 1, Born grids at spacing 0.5 (3D).
def _dims(case):
    return tuple(int(v) for v in case["dims"].split("x"))


def _axis(lo, d, n):
    return lo + d * torch.arange(n, dtype=torch.float64, device="cuda")


def _rand(seed, *shape):
    g = torch.Generator()
    g.manual_seed(seed)
    return torch.rand(*shape, generator=g, dtype=torch.float64)


_DX1, _DX2 = 0.1, 0.3


def _inputs_1d(case, seed):
    n, L = case["n"], 0.5 * _DX1 * case["n"]
    x = _axis(-L, _DX1, n)
    out = []
    for c in range(case["count"]):
        r = _rand(1000003 * seed + c, 6).tolist()
        s, x0, k = 0.06 * L + 0.04 * L * r[0], L * (-0.5 + 0.3 * r[1]), 0.5 + r[2]
        psi = torch.exp(-(x - x0) ** 2 / (4 * s * s)) * torch.exp(1j * k * x)
        psi = psi / torch.sqrt((psi.abs() ** 2).sum() * _DX1)
        V = (0.2 + r[3]) * torch.exp(-(x - 0.2 * L * r[4]) ** 2 / (2 * (0.5 + r[5]) ** 2))
        out.append((psi, V.to(torch.complex128)))
    return L, out


_DT1 = 0.05
_DT2 = 0.1


def _inputs_2d(case, seed):
    nx, ny = case["nx"], case["ny"]
    Lx, Ly = 0.5 * _DX2 * nx, 0.5 * _DX2 * ny
    X, Y = _axis(-Lx, _DX2, nx)[:, None], _axis(-Ly, _DX2, ny)[None, :]
    out = []
    for c in range(case["count"]):
        r = _rand(1000003 * seed + c, 64).tolist()
        sx, sy = 0.08 * Lx, 0.08 * Ly
        psi = (torch.exp(1j * (0.5 + r[0]) * X - (X + 0.4 * Lx) ** 2 / (4 * sx * sx)) *
               torch.exp(1j * (r[1] - 0.5) * Y - Y ** 2 / (4 * sy * sy)))
        psi = psi / torch.sqrt((psi.abs() ** 2).sum() * _DX2 * _DX2)
        V = torch.zeros(nx, ny, dtype=torch.float64, device="cuda")
        for b in range(12):
            h, w, cx, cy = r[4 * b + 4:4 * b + 8]
            w = 1.0 + 3.0 * w
            V += h * (torch.exp(-(X - 0.6 * Lx * (cx - 0.5)) ** 2 / (2 * w * w)) *
                      torch.exp(-(Y - Ly * (cy - 0.5)) ** 2 / (2 * w * w)))
        V = V.to(torch.complex128)
        if case["absorb"]:
            wd = 0.1 * min(Lx, Ly)
            d = torch.minimum(torch.minimum(X + Lx, Lx - X).expand(nx, ny),
                              torch.minimum(Y + Ly, Ly - Y).expand(nx, ny))
            V = V - 1j * torch.where(d < wd, 0.1 * ((wd - d) / wd) ** 2, torch.zeros_like(d))
        out.append((psi, V))
    return Lx, Ly, out


def _inputs_fft(case, seed):
    dims = _dims(case)
    r = 2 * _rand(1000003 * seed + 5, *dims, 2).cuda() - 1
    z = torch.view_as_complex(r)
    return z if case["precision"] == 64 else z.to(torch.complex64)


def _born_setup(case, seed):
    """Half widths of the box, the energies and the physical potential.  2D
    boxes hold the 24 wavelengths that the preconditioned solver asks for,
    3D boxes its 20 / k."""
    dims = _dims(case)
    r = _rand(1000003 * seed + 9, 80).tolist()
    if len(dims) == 2:
        d = 0.5
        half = [0.5 * d * n for n in dims]
        kmin = 1.02 * 24 * 2 * math.pi / (2 * min(half))
        ks = [kmin * (1.0 + 0.3 * r[i]) for i in range(case["energies"])]
        # at most a phase of 2 per grid step
        ks = [min(k, 4.0) for k in ks]
    else:
        d = 0.5
        half = [0.5 * d * n for n in dims]
        kmin = 1.02 * 20 / (2 * min(half))
        ks = [kmin + (max(kmin, 2.0) - kmin + 0.5) * r[i] for i in range(case["energies"])]
    ax = [_axis(-h, d, n) for h, n in zip(half, dims)]
    V = torch.zeros(dims, dtype=torch.float64, device="cuda")
    for b in range(8):
        a, w = 0.3 * r[20 + 6 * b], 1.5 + 2.5 * r[21 + 6 * b]
        t = a
        for i, x in enumerate(ax):
            c = 0.6 * half[i] * (r[22 + 6 * b + i] - 0.5)
            e = torch.exp(-(x - c) ** 2 / (2 * w * w))
            t = t * e.reshape([-1 if q == i else 1 for q in range(len(dims))])
        V += t
    return half, [0.5 * k * k for k in ks], V.to(torch.complex128), d


# ------------------------------------------------------- prepare and run
class _View:
    """A device buffer of the package as an array that torch can wrap."""

    def __init__(self, buf):
        self._buf = buf
        self.__cuda_array_interface__ = {
            "shape": buf.shape, "typestr": buf.dtype.str, "data": (int(buf.ptr), False),
            "version": 3, "strides": None}


def _tensor(buf, shape):
    return torch.as_tensor(_View(buf), device="cuda").reshape(shape)


def _method(order):
    return SolverMethod.SplittingMethodO2 if order == 2 else SolverMethod.SplittingMethodO4


def prepare(case, seed):
    kind = case["kind"]
    if kind == "evolve1d":
        L, items = _inputs_1d(case, seed)
        evs = []
        for psi, V in items:
            o = Options().Hip().Batch(case["steps"]).Precision(case["precision"])
            b = BoundaryCondition.InfiniteWall if case["wall"] else BoundaryCondition.Period
            evs.append(Evolver1D().init(psi.cpu().numpy(), False, _DT1, False, V.cpu().numpy(),
                                        -L, L, case["n"], b, _method(case["order"]), 1.0, 1.0, o))
        return dict(case=case, evs=evs, psi=[_tensor(e.psi, (case["n"],)) for e in evs])
    if kind == "evolve2d":
        Lx, Ly, items = _inputs_2d(case, seed)
        evs = []
        for psi, V in items:
            o = Options().Hip().Batch(case["steps"]).Precision(case["precision"])
            o.ComplexPotential(case["absorb"])
            evs.append(Evolver2D().init(psi.cpu().numpy(), False, _DT2, False, V.cpu().numpy(),
                                        -Lx, Lx, case["nx"], -Ly, Ly, case["ny"],
                                        BoundaryCondition.Period, _method(case["order"]), 1.0,
                                        1.0, o))
        return dict(case=case, evs=evs,
                    psi=[_tensor(e.psi, (case["nx"], case["ny"])) for e in evs])
    if kind == "fft":
        dims, p = _dims(case), case["precision"]
        x = _inputs_fft(case, seed)
        return dict(case=case, x=x, y=torch.empty_like(x), z=torch.empty_like(x),
                    fwd=FourierTransform(dims, False, p), inv=FourierTransform(dims, True, p))
    half, E, V, d = _born_setup(case, seed)
    dims = _dims(case)
    o = Options().Hip().Order(case["iters"]).Preconditional(True).Slow(0.5)
    o.SetString("preconditioner", case["pre"]).Precision(case["precision"])
    V = V.cpu().numpy()
    if len(dims) == 2:
        s = QuPerturbation2D().init(V, -half[0], half[0], dims[0], -half[1], half[1], dims[1], E,
                                    0.0, 1.0, 0.0, SolverMethod.BornSerise, 1.0, 1.0, o)
    else:
        s = QuPerturbation3D().init(V, -half[0], half[0], dims[0], -half[1], half[1], dims[1],
                                    -half[2], half[2], dims[2], E, 0.0, 0.0, 0.0, 1.0,
                                    SolverMethod.BornSerise, 1.0, 1.0, o)
    out = [torch.empty(dims, dtype=torch.complex128, device="cuda") for _ in E]
    return dict(case=case, solver=s, out=out)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("evolve1d", "evolve2d"):
        evs = state["evs"]
        if len(evs) == 1:
            evs[0].step()
        else:
            advance_batched(evs, case["steps"])
        if case.get("norm"):
            return state["psi"] + [evs[0].Norm2()]
        return state["psi"]
    if kind == "fft":
        state["fwd"].transform(state["x"].data_ptr(), state["y"].data_ptr())
        state["inv"].transform(state["y"].data_ptr(), state["z"].data_ptr())
        return [state["y"], state["z"]]
    s = state["solver"]
    s.Compute()
    for e, out in enumerate(state["out"]):
        N.call("qsim_hip_born_get_dpsi", s._job, e, ctypes.c_void_p(out.data_ptr()), None)
    fwd = (1.0, 0.0) if out.dim() == 2 else (0.0, 0.0, 1.0)
    return state["out"] + [s.ComputeXSection(*fwd)]


def work(case):
    kind = case["kind"]
    if kind == "fft":
        n = math.prod(_dims(case))
        es = 16 if case["precision"] == 64 else 8
        return {"bytes": 4 * n * es, "flops": 2 * 5 * n * math.log2(n)}
    if kind == "born":
        n, k = math.prod(_dims(case)), case["energies"]
        # the potential once, each energy's result once; per iteration two
        # transforms, the source, the Green's function and the update
        return {"bytes": n * 16 + k * n * 16,
                "flops": k * case["iters"] * n * (2 * 5 * math.log2(n) + 50)}
    n = case["n"] if kind == "evolve1d" else case["nx"] * case["ny"]
    stages = case["steps"] * (1 if case["order"] == 2 else 3)
    m = 2 * n if case.get("wall") else n
    vbytes = 16 if case.get("absorb") else 8
    return {"bytes": case["count"] * n * (32 + vbytes),
            "flops": case["count"] * stages * (2 * 5 * m * math.log2(m) + 12 * n)}


# ----------------------------------------------------- the same in 64 bits
def _fold(n, dk):
    i = torch.arange(n, dtype=torch.float64, device="cuda")
    return torch.where(i > n // 2, n - i, i) * dk


def _stages(order):
    """(potential weight, kinetic weight) pairs and the closing weight."""
    if order == 2:
        return [(0.5, 1.0)], 0.5
    c1, c2 = 1 / (2 * (2 - _O4_T)), (1 - _O4_T) / (2 * (2 - _O4_T))
    d1, d2 = 1 / (2 - _O4_T), -_O4_T / (2 - _O4_T)
    return [(c1, d1), (c2, d2), (c2, d1)], c1


def _split(psi, V, T, dt, order, steps, apply_t):
    st, end = _stages(order)
    for _ in range(steps):
        for cv, ct in st:
            psi = apply_t(torch.exp(-1j * dt * cv * V) * psi, torch.exp(-1j * dt * ct * T))
        psi = torch.exp(-1j * dt * end * V) * psi
    return psi


def _sine(a, f):
    """Odd extension, transform, factor, and back."""
    n = a.shape[0]
    z = torch.zeros(1, dtype=a.dtype, device=a.device)

    def odd(u):
        return torch.cat([z, u[1:], z, -u[1:].flip(0)])
    b = torch.fft.ifft(odd(a), norm="forward")
    g = b[:n] * f
    return -torch.fft.ifft(odd(g), norm="forward")[:n] / (2 * n)


def _exact_born(case, seed):
    half, energies, V, d = _born_setup(case, seed)
    dims = _dims(case)
    dim = len(dims)
    shape = [[-1 if q == i else 1 for q in range(dim)] for i in range(dim)]
    out, first = [], None
    for E in energies:
        k0 = math.sqrt(2 * E)
        ab = 0
        psi0 = 1.0
        T = 0
        for i, n in enumerate(dims):
            j = torch.arange(n, device="cuda")
            x = torch.where(j < n // 2, j, n - j).double() * d * k0
            u = 1 - x * x / 225.0
            lay = torch.where(u > 0, torch.exp(-0.015 * x * x /
                                               torch.sqrt(torch.clamp(u, min=1e-300))),
                              torch.zeros_like(x))
            ab = ab + (-0.8 * E * lay).reshape(shape[i])
            if i == (0 if dim == 2 else 2):
                psi0 = torch.exp(1j * k0 * _axis(-half[i], d, n)).reshape(shape[i])
            T = T + (0.5 * _fold(n, 2 * math.pi / (n * d)) ** 2).reshape(shape[i])
        Ve = V + 1j * ab
        eps = Ve.abs().max().item()
        g0 = 1.0 / torch.complex(E - T, torch.full_like(T, eps))
        gam = 0.5 * (1 - 1j * (Ve.conj() if case["pre"] == "Hao1" else Ve) / eps)
        if case["pre"] == "Hao2":
            gam = 0.5 * 2 / (1 + 1j * Ve / eps)
        src = torch.complex(Ve.real, Ve.imag + eps)
        dp = torch.zeros(dims, dtype=torch.complex128, device="cuda")
        for _ in range(case["iters"]):
            t = torch.fft.ifftn(g0 * torch.fft.fftn(src * dp + Ve.real * psi0))
            dp = (1 - gam) * dp + gam * t
        out.append(dp)
        if first is None:
            r = ((psi0 + dp) * V.real * torch.conj(psi0)).sum().item()
            if dim == 3:
                first = abs(r * 2 * d ** 3 / (4 * math.pi)) ** 2
            else:
                first = abs(r * 2 * d * d / 4) ** 2 * 2 / (math.pi * k0)
    return out + [first]


def exact(case, seed):
    kind = case["kind"]
    if kind == "fft":
        x = _inputs_fft(case, seed).to(torch.complex128)
        return [torch.fft.fftn(x), x * x.numel()]
    if kind == "born":
        return _exact_born(case, seed)
    if kind == "evolve1d":
        L, items = _inputs_1d(case, seed)
        n, res = case["n"], []
        for psi, V in items:
            if case["wall"]:
                k = torch.arange(n, dtype=torch.float64, device="cuda") * math.pi / (_DX1 * n)
                go = _sine
            else:
                k = _fold(n, 2 * math.pi / (_DX1 * n))

                def go(a, f):
                    return torch.fft.ifft(torch.fft.fft(a) * f)
            res.append(_split(psi, V, 0.5 * k * k, _DT1, case["order"], case["steps"], go))
        if case["norm"]:
            res.append(((res[0].abs() ** 2).sum() * _DX1).item())
        return res
    Lx, Ly, items = _inputs_2d(case, seed)
    kx = _fold(case["nx"], 2 * math.pi / (_DX2 * case["nx"]))
    ky = _fold(case["ny"], 2 * math.pi / (_DX2 * case["ny"]))
    T = 0.5 * (kx * kx)[:, None] + 0.5 * (ky * ky)[None, :]
    return [_split(psi, V, T, _DT2, case["order"], case["steps"],
                   lambda a, f: torch.fft.ifft2(torch.fft.fft2(a) * f)) for psi, V in items]
