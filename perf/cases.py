"""Measured workloads: what a program built on helmholtz_amd has the GPU do,
through the package's entry points and its C interface.

Kinds
-----
``apply``     Y = H X on device-resident blocks (``HelmholtzOperator.apply``):
              the outer product of a user's own Krylov or time-harmonic loop.
``apply_ho``  the same for the spread operator (``GetHelmholtzOperatorHO``).
``cycle``     Z = M^-1 V, one multigrid cycle as the preconditioner of a user's
              own Krylov method (``hh_solver_precondition`` on device blocks).
``solve``     ``solveLinearSystem`` with a kept solver and new right-hand sides:
              one source per call or many, plain or mixed precision.
``fwi``       one frequency of a waveform-inversion step on a new model: the
              operator, the solver, a forward and an adjoint solve from host
              arrays, nothing kept from the model before.
``unet``      loss and gradient of the coarse-grid correction network on one
              training batch.

Media are the package's seeded layered-plus-body generators (1500-4500 m/s,
h = 10 m), frequencies 8-12 points per wavelength, point sources near the top,
as in the repository's benchmark and tests.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "helmholtz.jl_amd"))

import helmholtz_amd as ha  # noqa: E402
from helmholtz_amd import _lib, learned, media  # noqa: E402
from helmholtz_amd.device import DeviceArray  # noqa: E402

H0 = 10.0


def listed():
    return [
        # one product on a small grid: a single-source loop, bound by the call itself
        {"name": "apply2d_small", "kind": "apply", "n1": 129, "n2": 129, "n3": 0, "nrhs": 1, "prec": "c128"},
        # the product over a 3-D survey's wavefields in mixed precision
        {"name": "apply3d_large", "kind": "apply", "n1": 193, "n2": 193, "n3": 97, "nrhs": 32, "prec": "c64"},
        # the spread operator on an odd 3-D grid, a few wavefields
        {"name": "apply_ho3d", "kind": "apply_ho", "n1": 101, "n2": 83, "n3": 57, "nrhs": 8, "beta": 0.8},
        # the benchmark's 2-D survey: 256 wavefields preconditioned at once, complex64
        {"name": "cycle2d_batch", "kind": "cycle", "n1": 1025, "n2": 513, "n3": 0, "nrhs": 256, "prec": "c64",
         "cycle": "W", "levels": 6, "wlevels": 3, "ppw": 8.0},
        # the 3-D survey's preconditioner, complex64
        {"name": "cycle3d_batch", "kind": "cycle", "n1": 193, "n2": 193, "n3": 97, "nrhs": 32, "prec": "c64",
         "cycle": "W", "levels": 5, "wlevels": 0, "ppw": 8.0},
        # the plain method on the small workload: one source, complex128 throughout
        {"name": "solve2d_small", "kind": "solve", "n1": 129, "n2": 129, "n3": 0, "nrhs": 1, "prec": "c128",
         "cycle": "V", "levels": 3, "wlevels": 0, "ppw": 10.0, "relax": "Jac", "krylov": "GMRES", "inner": 10,
         "tol": 1e-6},
        # the plain method on the benchmark's grid, one source per call
        {"name": "solve2d_plain", "kind": "solve", "n1": 1025, "n2": 513, "n3": 0, "nrhs": 1, "prec": "c128",
         "cycle": "W", "levels": 6, "wlevels": 3, "ppw": 8.0, "relax": "Jac", "krylov": "GMRES", "inner": 10,
         "tol": 1e-6},
        # many sources at once, mixed precision, solved tightly (gradient checks, reference wavefields)
        {"name": "solve2d_batch", "kind": "solve", "n1": 1025, "n2": 513, "n3": 0, "nrhs": 48, "prec": "c64",
         "cycle": "W", "levels": 6, "wlevels": 3, "ppw": 8.0, "relax": "Jac", "krylov": "GMRES", "inner": 10,
         "tol": 1e-12},
        # a 3-D shot gather in complex128
        {"name": "solve3d_plain", "kind": "solve", "n1": 97, "n2": 97, "n3": 49, "nrhs": 8, "prec": "c128",
         "cycle": "W", "levels": 4, "wlevels": 0, "ppw": 8.0, "relax": "Jac", "krylov": "GMRES", "inner": 8,
         "tol": 1e-6},
        # the reference test's K-cycle with Jac-GMRES smoothing, a few sources
        {"name": "solve2d_kcycle", "kind": "solve", "n1": 257, "n2": 129, "n3": 0, "nrhs": 4, "prec": "c128",
         "cycle": "K", "levels": 3, "wlevels": 0, "ppw": 10.0, "relax": "Jac-GMRES", "krylov": "GMRES", "inner": 5,
         "tol": 1e-6},
        # one frequency of an inversion step: new model, forward and adjoint solves from host arrays
        {"name": "fwi_step", "kind": "fwi", "n1": 257, "n2": 129, "n3": 0, "nrhs": 4, "prec": "c128", "cycle": "W",
         "levels": 3, "wlevels": 0, "ppw": 10.0, "relax": "Jac", "krylov": "GMRES", "inner": 10, "tol": 1e-6},
        # a training batch of the correction network at the size it is trained at
        {"name": "unet_batch", "kind": "unet", "n1": 129, "n2": 129, "images": 16},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _coarsenable(rng, lo, hi, levels):
    """A node count 2^(levels-1) k + 1 in about [lo, hi] (k odd or even)."""
    s = 2 ** (levels - 1)
    return s * max(2, int(round(_log_int(rng, lo, hi) / s))) + 1


def draw(rng):
    kind = rng.choice(["apply", "apply", "apply_ho", "cycle", "cycle", "solve", "solve", "solve", "fwi", "unet"])
    if kind in ("apply", "apply_ho"):
        prec = "c128" if kind == "apply_ho" else rng.choice(["c128", "c64"])
        most = (8 if kind == "apply_ho" else 48) << 20
        if rng.random() < 0.5:
            n = (_log_int(rng, 33, 1200), _log_int(rng, 33, 1200), 0)
            nodes = n[0] * n[1]
        else:
            n = (_log_int(rng, 17, 200), _log_int(rng, 17, 200), _log_int(rng, 17, 120))
            nodes = n[0] * n[1] * n[2]
        c = {"kind": kind, "n1": n[0], "n2": n[1], "n3": n[2], "nrhs": _log_int(rng, 1, max(1, min(256, most // nodes)))}
        c.update({"beta": round(rng.uniform(0.5, 1.0), 2)} if kind == "apply_ho" else {"prec": prec})
        return c
    if kind == "unet":
        return {"kind": kind, "n1": 8 * rng.randint(4, 24) + 1, "n2": 8 * rng.randint(4, 24) + 1,
                "images": rng.randint(1, 16)}
    if kind == "cycle":
        prec = rng.choice(["c64", "c64", "c128"])
        if rng.random() < 0.6:
            levels = rng.choice([3, 4, 5])
            n = (_coarsenable(rng, 129, 1025, levels), _coarsenable(rng, 65, 513, levels), 0)
            while (n[0] >> (levels - 1)) * (n[1] >> (levels - 1)) > 1500:
                levels += 1
                n = tuple(((v - 1) >> (levels - 1) << (levels - 1)) + 1 for v in n[:2]) + (0,)
            nodes = n[0] * n[1]
        else:
            levels = rng.choice([3, 4])
            n = (_coarsenable(rng, 49, 145, levels), _coarsenable(rng, 49, 145, levels), _coarsenable(rng, 33, 81, levels))
            while (n[0] >> (levels - 1)) * (n[1] >> (levels - 1)) * (n[2] >> (levels - 1)) > 900:
                levels += 1
                n = tuple(max(2, (v - 1) >> (levels - 1)) * (1 << (levels - 1)) + 1 for v in n)
            nodes = n[0] * n[1] * n[2]
        return {"kind": kind, "n1": n[0], "n2": n[1], "n3": n[2], "prec": prec,
                "nrhs": _log_int(rng, 1, max(1, min(128, (32 << 20) // nodes))), "cycle": rng.choice(["V", "W", "W"]),
                "levels": levels, "wlevels": rng.choice([0, 2]), "ppw": round(rng.uniform(8.0, 12.0), 2)}
    c = {"kind": kind, "prec": "c128", "wlevels": 0, "ppw": round(rng.uniform(10.0, 12.0), 2), "relax": "Jac",
         "krylov": "GMRES", "inner": rng.choice([8, 10, 12]), "tol": 1e-6, "cycle": "W"}
    if kind == "fwi":
        c.update({"n1": _coarsenable(rng, 97, 321, 3), "n2": _coarsenable(rng, 65, 161, 3), "n3": 0,
                  "nrhs": rng.randint(1, 8), "levels": 3})
        return c
    shape = rng.choice(["plain", "plain", "batch", "3d", "kcycle"])
    if shape == "3d":
        c.update({"n1": _coarsenable(rng, 33, 81, 3), "n2": _coarsenable(rng, 33, 81, 3), "n3": _coarsenable(rng, 25, 41, 3),
                  "levels": 3, "nrhs": rng.randint(1, 8)})
    elif shape == "kcycle":
        c.update({"n1": _coarsenable(rng, 97, 321, 3), "n2": _coarsenable(rng, 65, 161, 3), "n3": 0, "levels": 3,
                  "nrhs": rng.randint(1, 6), "cycle": "K", "relax": "Jac-GMRES", "inner": 5})
    else:
        c.update({"n1": _coarsenable(rng, 129, 513, 4), "n2": _coarsenable(rng, 97, 257, 4), "n3": 0, "levels": 4,
                  "nrhs": 1 if shape == "plain" else rng.randint(8, 64)})
        if shape == "batch":
            c.update({"prec": "c64", "tol": 1e-12})
    return c


# ------------------------------------------------------------------ inputs
def _nodes(c):
    return [c["n1"], c["n2"]] + ([c["n3"]] if c.get("n3") else [])


def _problem(c, seed):
    """Mesh, squared slowness, attenuation without the absorbing layer, frequency."""
    n = _nodes(c)
    v = (media.layered_body_velocity_2d if len(n) == 2 else media.layered_body_velocity_3d)(tuple(n), seed=seed % 65521)
    m = (1.0 / v**2).ravel(order="F")
    mesh = ha.getRegularMesh([x for k in n for x in (0.0, H0 * (k - 1))], [k - 1 for k in n])
    w = media.omega_for_ppw(1500.0, H0, c.get("ppw", 10.0))
    return mesh, m, 0.01 * w * np.ones(m.size), w


def _pad(n):
    return [max(2, min(20, k // 8)) for k in n]


def _param(c, seed):
    mesh, m, g, w = _problem(c, seed)
    n = _nodes(c)
    g = g + ha.getABL(n, True, _pad(n), w).ravel(order="F")
    return ha.HelmholtzParam(mesh, g, m, w, True, True)


def _subscripts(c, seed):
    """1-based source subscripts near the top, spread over the survey."""
    n, rng = _nodes(c), np.random.default_rng(seed)
    lo = [max(2, k // 10) for k in n[:-1]]
    return [tuple(int(rng.integers(a, k - a)) for a, k in zip(lo, n[:-1])) + (int(rng.integers(2, 5)),)
            for _ in range(c["nrhs"])]


class _Block:
    """A DeviceArray seen by torch (no copy; keeps the block alive)."""

    def __init__(self, a):
        self.a = a
        real = "<f8" if a.dtype == np.complex128 else "<f4"
        ncol = a.shape[1] if len(a.shape) > 1 else 1
        self.__cuda_array_interface__ = {"shape": (ncol, a.shape[0], 2), "typestr": real, "data": (a.ptr, False),
                                         "version": 2}


def _torch(a):
    return torch.as_tensor(_Block(a), device="cuda")


def _random_values(c, seed, dtype):
    """nrhs x N standard-normal complex values (torch, on the GPU)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    N = math.prod(_nodes(c))
    return torch.randn((c["nrhs"], N, 2), dtype=dtype, device="cuda", generator=gen)


def _random_block(c, seed, prec):
    dt, td = (np.complex128, torch.float64) if prec == "c128" else (np.complex64, torch.float32)
    X = DeviceArray((math.prod(_nodes(c)), c["nrhs"]), dt)
    _torch(X).copy_(_random_values(c, seed, td))
    return X


def _mg(c):
    mg = ha.getMGparam(complex, int, c["levels"], 1, 400, c.get("tol", 1e-6), c.get("relax", "Jac"), 0.8, 2, 2,
                       c["cycle"], "NoMUMPS", 0.5, 0.0)
    mg.prec = c["prec"]
    mg.wlevels = c["wlevels"]
    return mg


def _solver(c, param):
    return ha.getShiftedLaplacianMultigridSolver(param, _mg(c), 0.5, c.get("krylov", "GMRES"), c.get("inner", 1))


def _features(c, seed):
    """Network inputs as the solver forms them (a scaled residual, k^2 h^2 and
    gamma / w, smooth in space) and targets of the corrections' size."""
    rng = np.random.default_rng(seed)
    n1, n2, im = c["n1"], c["n2"], c["images"]
    X, Z = np.meshgrid(np.linspace(0, 1, n1), np.linspace(0, 1, n2), indexing="ij")

    def wave(k):
        a, b, p = rng.uniform(-k, k), rng.uniform(-k, k), rng.uniform(0, 2 * np.pi)
        return np.cos(2 * np.pi * (a * X + b * Z) + p)

    f = np.empty((im, n1 * n2, 4), np.float32)
    t = np.empty((im, n1 * n2, 2), np.float32)
    for q in range(im):
        ph = sum(wave(20) for _ in range(6)) / 1.7
        f[q, :, 0] = (ph + 0.1 * rng.standard_normal(X.shape)).ravel(order="F")
        f[q, :, 1] = (sum(wave(20) for _ in range(6)) / 1.7).ravel(order="F")
        f[q, :, 2] = (1.5 + 0.8 * wave(2)).ravel(order="F")
        f[q, :, 3] = (0.01 + np.maximum(0.0, np.abs(X - 0.5) - 0.4) ** 2 * 100).ravel(order="F")
        t[q, :, 0] = (0.3 * ph).ravel(order="F")
        t[q, :, 1] = (0.3 * wave(10)).ravel(order="F")
    return f, t


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind, "case": case}
    if kind == "unet":
        s["net"] = learned.UNet(seed=seed % 1000003)
        s["feats"], s["target"] = _features(case, seed)
        return s
    if kind == "fwi":
        s["mesh"], s["m"], s["gamma"], s["omega"] = _problem(case, seed)
        s["B"] = ha.point_sources(s["mesh"], _subscripts(case, seed))
        rng = np.random.default_rng(seed + 1)
        rec = np.zeros_like(s["B"])  # data residual on a line of receivers
        n1 = case["n1"]
        row = slice(2 * n1 + n1 // 10, 3 * n1 - n1 // 10)
        rec[row] = rng.standard_normal(rec[row].shape) + 1j * rng.standard_normal(rec[row].shape)
        s["residual"] = rec
        return s
    p = _param(case, seed)
    if kind == "apply":
        s["H"] = ha.GetHelmholtzOperator(p)
    elif kind == "apply_ho":
        s["H"] = ha.GetHelmholtzOperatorHO(p, case["beta"])
    if kind in ("apply", "apply_ho"):
        s["prec"] = case.get("prec", "c128")
        s["X"] = _random_block(case, seed, s["prec"])
        s["Y"] = s["X"].empty_like()
        s["out"] = _torch(s["Y"])
        return s
    s["solver"] = _solver(case, p)
    if kind == "cycle":
        s["V"] = _random_block(case, seed, "c128")
        s["Z"] = DeviceArray(s["V"].shape, np.complex64 if case["prec"] == "c64" else np.complex128)
        s["out"] = _torch(s["Z"])
        s["solver"].MG.relativeTol = 1e-6
        from helmholtz_amd.solver import _ensure_handle
        _ensure_handle(s["solver"])
    else:
        s["B"] = DeviceArray.from_numpy(ha.point_sources(p.Mesh, _subscripts(case, seed)))
    return s


def run(state):
    kind = state["kind"]
    if kind in ("apply", "apply_ho"):
        state["H"].apply(state["X"], state["prec"], out=state["Y"])
        return state["out"]
    if kind == "cycle":
        _lib.check(_lib.lib().hh_solver_precondition(state["solver"]._handle, state["V"].ptr, state["Z"].ptr,
                                                     state["V"].shape[1], _lib.HH_DEVICE))
        return state["out"]
    if kind == "solve":
        X, _ = ha.solveLinearSystem(None, state["B"], state["solver"])
        return _torch(X)
    if kind == "fwi":
        c = state["case"]
        n = _nodes(c)
        w = state["omega"]
        H, g = ha.GetHelmholtzOperator(state["mesh"], state["m"], w, state["gamma"], True, _pad(n), w, True)
        solver = _solver(c, ha.HelmholtzParam(state["mesh"], g.ravel(order="F"), state["m"], w, True, True))
        u, solver = ha.solveLinearSystem(H, state["B"], solver)
        adj, solver = ha.solveLinearSystem(H, state["residual"], solver, 1)
        return {"u": u, "adjoint": adj}
    loss, grad = state["net"].loss_grad(state["feats"], state["target"], state["case"]["n1"], state["case"]["n2"])
    return {"loss": loss, "grad": grad}


def work(case):
    """Inputs read once and outputs written once, and the arithmetic of one
    pass; for a solve, whose iteration count depends on the model, its data."""
    kind = case["kind"]
    if kind == "unet":
        px = case["n1"] * case["n2"] * case["images"]
        macs = 9 * (2 * 16 * 16 + (16 * 32 + 32 * 32) / 4 + (32 * 64 + 64 * 64) / 16 + 2 * 64 * 64 / 64
                    + (128 * 64 + 64 * 64) / 16 + (96 * 32 + 32 * 32) / 4 + 48 * 16 + 16 * 16) + 32
        return {"bytes": px * 24.0 + 8.0 * 304738, "flops": 3 * 2.0 * macs * px}
    N = math.prod(_nodes(case))
    a = N * case["nrhs"]
    if kind == "apply":
        v = 16 if case["prec"] == "c128" else 8
        return {"bytes": 2.0 * v * a + v * N, "flops": (24.0 if case.get("n3") else 18.0) * a}
    if kind == "apply_ho":
        return {"bytes": 32.0 * a + 16 * N, "flops": (19 * 4 + 7 * 8.0 if case.get("n3") else 9 * 4 + 5 * 8.0) * a}
    if kind == "cycle":
        v = 8 if case["prec"] == "c64" else 16
        fine = 4 * 14.0 + (2 if case["cycle"] == "W" else 1) * 30.0
        return {"bytes": (16.0 + v) * a + 2 * v * N, "flops": 1.3 * fine * a}
    return {"bytes": (32.0 if kind == "solve" else 64.0) * a + 16 * N, "flops": 100.0 * a}


# ------------------------------------------------------------------ 64-bit values
def _axis(t, axis, dim):
    """Torch dimension of grid axis ``axis`` in an array (..., [n3,] n2, n1)."""
    return t.dim() - 1 - axis


def _take(t, d, i):
    return t.index_select(d, i)


def _second_difference(x, axis, ih):
    """sum of ih (2 x - x_lo - x_hi) along a grid axis, mirrored at both ends."""
    d = x.dim() - 1 - axis
    n = x.shape[d]
    lo = torch.arange(n, device=x.device) - 1
    hi = lo + 2
    lo[0], hi[-1] = 1, n - 2
    return ih * (2 * x - x.index_select(d, lo) - x.index_select(d, hi))


def _diagonal(n, h, m, gamma, w):
    """-w^2 m (1 - i gamma / w) and the Sommerfeld terms (Neumann top), torch complex128 (..., n2, n1)."""
    shape = tuple(reversed(n))
    m = torch.as_tensor(np.asarray(m, dtype=np.float64), device="cuda").reshape(shape)
    g = torch.as_tensor(np.asarray(gamma, dtype=np.float64), device="cuda").reshape(shape)
    d = torch.complex(-(w * w) * m, w * g * m)
    for axis in range(len(n)):
        t = d.dim() - 1 - axis
        s = torch.zeros(n[axis], dtype=torch.float64, device="cuda")
        s[-1] += 2.0 / h[axis]
        if axis != len(n) - 1:
            s[0] += 2.0 / h[axis]
        d = d + 1j * w * torch.sqrt(m) * s.reshape([-1 if k == t else 1 for k in range(d.dim())])
    return d


def _helmholtz(x, d, h):
    y = d * x
    for axis in range(len(h)):
        y = y + _second_difference(x, axis, 1.0 / h[axis] ** 2)
    return y


def _tridiagonal(x, axis, lo, di, up):
    """Rows (lo_i, di_i, up_i) of a symmetric-structure tridiagonal along a grid axis."""
    d = x.dim() - 1 - axis
    n = x.shape[d]
    view = [-1 if k == d else 1 for k in range(x.dim())]
    y = di.reshape(view) * x
    y.narrow(d, 1, n - 1).add_(lo[1:].reshape([-1 if k == d else 1 for k in range(x.dim())]) * x.narrow(d, 0, n - 1))
    y.narrow(d, 0, n - 1).add_(up[:-1].reshape([-1 if k == d else 1 for k in range(x.dim())]) * x.narrow(d, 1, n - 1))
    return y


def _average(x, axis, a):
    n = x.shape[x.dim() - 1 - axis]
    o = torch.full((n,), (1 - a) / 2, dtype=torch.float64, device=x.device)
    di = torch.full((n,), a, dtype=torch.float64, device=x.device)
    di[0] = di[-1] = 0.5 + a / 2
    return _tridiagonal(x, axis, o, di, o)


def _natural(x, axis, ih):
    n = x.shape[x.dim() - 1 - axis]
    o = torch.full((n,), -ih, dtype=torch.float64, device=x.device)
    di = torch.full((n,), 2 * ih, dtype=torch.float64, device=x.device)
    di[0] = di[-1] = ih
    return _tridiagonal(x, axis, o, di, o)


def _spread(x, d, h, beta):
    """The spread Laplacian plus the averaged mass (src/PlainNodalLaplacian.jl:69-141)."""
    dim = len(h)
    y = torch.zeros_like(x)
    for axis in range(dim):
        others = [q for q in range(dim) if q != axis]
        p = beta * x
        for q in others:
            p = p + (1 - beta) / len(others) * _average(x, q, 0.5)
        y = y + _natural(p, axis, 1.0 / h[axis] ** 2)
    dx = d * x
    for axis in range(dim):
        y = y + _average(dx, axis, beta) / dim
    return y


def _weigh(x, axis):
    """Full weighting along one axis (mirrored)."""
    d = x.dim() - 1 - axis
    n = x.shape[d]
    at = torch.arange(0, n, 2, device=x.device)
    lo, hi = at - 1, at + 1
    lo[0], hi[-1] = 1, n - 2
    return 0.5 * x.index_select(d, at) + 0.25 * (x.index_select(d, lo) + x.index_select(d, hi))


def _interpolate(x, axis):
    d = x.dim() - 1 - axis
    n = x.shape[d]
    shape = list(x.shape)
    shape[d] = 2 * n - 1
    y = x.new_empty(shape)
    y[tuple(slice(0, None, 2) if k == d else slice(None) for k in range(x.dim()))] = x
    y[tuple(slice(1, None, 2) if k == d else slice(None) for k in range(x.dim()))] = \
        0.5 * (x.narrow(d, 0, n - 1) + x.narrow(d, 1, n - 1))
    return y


class _Cycle:
    """One V or W cycle with two damped-Jacobi sweeps before and after."""

    def __init__(self, c, p):
        n, h = _nodes(c), [float(v) for v in p.Mesh.h]
        w = float(p.omega)
        m = torch.as_tensor(p.m, device="cuda").reshape(tuple(reversed(n)))
        g = torch.as_tensor(p.gamma, device="cuda").reshape(tuple(reversed(n))) + 0.5 * w
        self.c, self.lev = c, []
        for l in range(c["levels"]):
            d = _diagonal(n, h, m.cpu().numpy().ravel(), g.cpu().numpy().ravel(), w)
            self.lev.append((list(h), d, 0.8 / (d + sum(2.0 / v**2 for v in h))))
            if l + 1 < c["levels"]:
                for axis in range(len(n)):
                    m, g = _weigh(m, axis), _weigh(g, axis)
                n, h = [(k - 1) // 2 + 1 for k in n], [2 * v for v in h]
        h, d, _ = self.lev[-1]
        N = d.numel()
        eye = torch.eye(N, dtype=torch.complex128, device="cuda").reshape((N,) + tuple(d.shape))
        self.inv = torch.linalg.inv(_helmholtz(eye, d, h).reshape(N, N).T.contiguous())

    def __call__(self, b, l=0):
        h, d, f = self.lev[l]
        if l + 1 == len(self.lev):
            return (b.reshape(b.shape[0], -1) @ self.inv.T).reshape(b.shape)
        x = f * b
        x = x + f * (b - _helmholtz(x, d, h))
        w = self.c["cycle"] == "W" and (self.c["wlevels"] == 0 or l < self.c["wlevels"])
        for _ in range(2 if w else 1):
            r = b - _helmholtz(x, d, h)
            for axis in range(len(h)):
                r = _weigh(r, axis)
            e = self(r, l + 1)
            for axis in range(len(h)):
                e = _interpolate(e, axis)
            x = x + e
        for _ in range(2):
            x = x + f * (b - _helmholtz(x, d, h))
        return x


def _direct(d, h, B, adjoint=False):
    """H x = b (or H^H x = b) in 2-D by block elimination along the longer axis, refined once.
    d: (n2, n1); B: (nrhs, n2, n1)."""
    if d.shape[1] > d.shape[0]:
        return _direct(d.T, h[::-1], B.transpose(1, 2), adjoint).transpose(1, 2)
    no, ni = d.shape
    T = torch.zeros((ni, ni), dtype=torch.complex128, device=d.device)
    i = torch.arange(ni, device=d.device)
    ih = 1.0 / h[0] ** 2
    T[i, i] = 2 * ih + 2.0 / h[1] ** 2
    T[i[1:], i[1:] - 1] = -ih
    T[i[:-1], i[:-1] + 1] = -ih
    T[0, 1] = T[ni - 1, ni - 2] = -2 * ih
    up = torch.full((no,), -1.0 / h[1] ** 2, dtype=torch.float64)
    lo = up.clone()
    up[0] *= 2
    lo[-1] *= 2
    if adjoint:
        T, d = T.T.contiguous(), d.conj()
        up, lo = torch.cat([lo[1:], lo[:1]]), torch.cat([up[-1:], up[:-1]])
    S = []
    for k in range(no):
        A = T + torch.diag(d[k])
        if k:
            A = A - float(lo[k] * up[k - 1]) * S[-1]
        S.append(torch.linalg.inv(A))

    def solve(r):
        y = [r[:, 0]]
        for k in range(1, no):
            y.append(r[:, k] - float(lo[k]) * (y[-1] @ S[k - 1].T))
        x = [None] * no
        x[-1] = y[-1] @ S[-1].T
        for k in range(no - 2, -1, -1):
            x[k] = (y[k] - float(up[k]) * x[k + 1]) @ S[k].T
        return torch.stack(x, 1)

    def product(x):
        y = d * x + x @ T.T
        y[:, 1:] += lo[1:].reshape(-1, 1).to(d.device) * x[:, :-1]
        y[:, :-1] += up[:-1].reshape(-1, 1).to(d.device) * x[:, 1:]
        return y

    x = solve(B)
    return x + solve(B - product(x))


def _unet_exact(c, seed):
    f, t = _features(c, seed)
    th = torch.as_tensor(learned.UNet(seed=seed % 1000003).get_params(), device="cuda").double().requires_grad_(True)
    n1, n2, im = c["n1"], c["n2"], c["images"]
    at = [0]

    def part(k):
        at[0] += k
        return th[at[0] - k:at[0]]

    def conv(x, ci, co):
        W, b = part(9 * co * ci).reshape(9, co, ci), part(co)
        n, ny, nx, _ = x.shape
        xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
        y = b
        for q in range(9):
            y = y + xp[:, q // 3:q // 3 + ny, q % 3:q % 3 + nx] @ W[q].T
        return torch.relu(y)

    def down(x):
        xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
        xp = 0.25 * xp[:, :-2:2] + 0.5 * xp[:, 1:-1:2] + 0.25 * xp[:, 2::2]
        return 0.25 * xp[:, :, :-2:2] + 0.5 * xp[:, :, 1:-1:2] + 0.25 * xp[:, :, 2::2]

    def up(x):
        for d in (1, 2):
            n = x.shape[d]
            mid = 0.5 * (x.narrow(d, 0, n - 1) + x.narrow(d, 1, n - 1))
            both = torch.stack([x.narrow(d, 0, n - 1), mid], d + 1).flatten(d, d + 1)
            x = torch.cat([both, x.narrow(d, n - 1, 1)], d)
        return x

    x = torch.zeros((im, n2, n1, 16), dtype=torch.float64, device="cuda")
    x[..., :4] = torch.as_tensor(f, device="cuda").double().reshape(im, n2, n1, 4)
    s0 = conv(conv(x, 16, 16), 16, 16)
    s1 = conv(conv(down(s0), 16, 32), 32, 32)
    s2 = conv(conv(down(s1), 32, 64), 64, 64)
    b3 = conv(conv(down(s2), 64, 64), 64, 64)
    b4 = conv(conv(torch.cat([up(b3), s2], -1), 128, 64), 64, 64)
    b5 = conv(conv(torch.cat([up(b4), s1], -1), 96, 32), 32, 32)
    b6 = conv(conv(torch.cat([up(b5), s0], -1), 48, 16), 16, 16)
    hw, hb = part(32).reshape(2, 16), part(2)
    y = (b6 @ hw.T + hb).reshape(im, n1 * n2, 2)
    loss = ((y - torch.as_tensor(t, device="cuda").double()) ** 2).mean()
    loss.backward()
    return {"loss": float(loss.detach()), "grad": th.grad.detach()}


def _real(x):
    """(nrhs, ..., n2, n1) complex -> (nrhs, N, 2), the layout of the device blocks."""
    return torch.view_as_real(x.reshape(x.shape[0], -1).contiguous())


def _columns(x):
    """(nrhs, ..., n2, n1) complex -> numpy N x nrhs."""
    return np.ascontiguousarray(x.reshape(x.shape[0], -1).cpu().numpy().T)


def exact(case, seed):
    kind = case["kind"]
    if kind == "unet":
        return _unet_exact(case, seed)
    n = _nodes(case)
    shape = (case["nrhs"],) + tuple(reversed(n))
    if kind in ("solve", "fwi"):
        if len(n) == 3:
            return None  # no direct solve of a 3-D grid in the time there is
        p = _param(case, seed)
        h = [float(v) for v in p.Mesh.h]
        d = _diagonal(n, h, p.m, p.gamma, float(p.omega))
        B = torch.as_tensor(ha.point_sources(p.Mesh, _subscripts(case, seed)).T.copy(), device="cuda").reshape(shape)
        u = _direct(d, h, B)
        if kind == "solve":
            return _real(u)
        res = torch.as_tensor(prepare(case, seed)["residual"].T.copy(), device="cuda").reshape(shape)
        return {"u": _columns(u), "adjoint": _columns(_direct(d, h, res, True))}
    p = _param(case, seed)
    h = [float(v) for v in p.Mesh.h]
    if kind == "cycle":
        V = torch.view_as_complex(_random_values(case, seed, torch.float64)).reshape(shape)
        M = _Cycle(case, p)
        return _real(torch.cat([M(V[k:k + 32]) for k in range(0, V.shape[0], 32)]))
    td = torch.float64 if case.get("prec", "c128") == "c128" else torch.float32
    X = torch.view_as_complex(_random_values(case, seed, td).double()).reshape(shape)
    d = _diagonal(n, h, p.m, p.gamma, float(p.omega))
    if kind == "apply":
        return _real(_helmholtz(X, d, h))
    return _real(_spread(X, d, h, case["beta"]))
