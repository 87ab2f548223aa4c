"""Cases that time the work users have this framework do, through its public
entry points: driven solves (TM and TE, plain FP64 and mixed-precision
factors, one or several sources), adjoint gradients, frequency sweeps, mode
eigenproblems, shift-invert eigenfrequencies and modulated devices.

  listed()             the cases, as plain dicts
  draw(rng)            one more case of the same ranges
  prepare(case, seed)  what a user's program holds before the call
  run(state)           one pass
  work(case)           bytes and flops one pass cannot do without
  exact(case, seed)    the outputs in 64 bits, from scipy's sparse LU

Grids are dl = 0.02 um with absorbing boundaries at 1.55 um; the structures
are those of the benchmark: a design region of 8 x 8-cell pixels of
permittivity 1 or 12.25 between two guides, continuous designs for gradients,
rod lattices for eigenfrequencies and a phase-modulated guide.
"""
from __future__ import annotations

import ctypes as C
import logging
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "fdfd.jl_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "fdfd.jl_amd"))

import fdfd  # noqa: E402
from fdfd import _lib, adjoint, core, modes, modulated  # noqa: E402
from fdfd.solve import PRECISIONS, Engine  # noqa: E402

DL = 0.02                  # cell size, um
EPS0N = core.EPS0 * core.DEFAULT_L0
MU0N = core.MU0 * core.DEFAULT_L0
TOL = 1e-12                # relative residual asked for (the default of linsolve and gradients)


def listed():
    return [
        # A small driven solve through solve(device): the guide with a point
        # source that first-time users run (host arrays in and out).
        {"name": "solve_tm_200x120_fp64", "kind": "solve", "nx": 200, "ny": 120, "npml": 15,
         "pol": "TM", "precision": "fp64"},
        # The smallest call: a coupler of under 10,000 cells, as parameter
        # scans and unit tests of devices make by the thousand.
        {"name": "solve_te_96x80_mixed", "kind": "solve", "nx": 96, "ny": 80, "npml": 10,
         "pol": "TE", "precision": "mixed"},
        # The headline workload: permittivity and source resident on the GPU,
        # assemble + factor + refined solve + fields, mixed precision.
        {"name": "drive_tm_1024_mixed", "kind": "drive", "nx": 1024, "ny": 1024, "npml": 20,
         "pol": "TM", "precision": "mixed"},
        # The same with plain FP64 factors (the default precision).
        {"name": "drive_tm_1024_fp64", "kind": "drive", "nx": 1024, "ny": 1024, "npml": 20,
         "pol": "TM", "precision": "fp64"},
        # A ragged grid (odd on both sides, longer along x), TE.
        {"name": "drive_te_517x389_fp64", "kind": "drive", "nx": 517, "ny": 389, "npml": 13,
         "pol": "TE", "precision": "fp64"},
        # A ragged elongated grid, longer along y, TE, mixed.
        {"name": "drive_te_301x700_mixed", "kind": "drive", "nx": 301, "ny": 700, "npml": 16,
         "pol": "TE", "precision": "mixed"},
        # Inverse design: objective and gradient (forward solve, transposed
        # solve on the same factors, gradient kernel), host arrays.
        {"name": "gradient_1024x768_mixed", "kind": "gradient", "nx": 1024, "ny": 768, "npml": 20,
         "pol": "TM", "precision": "mixed"},
        # Resonances of a rod lattice: 8 eigenfrequencies by shift-invert
        # Arnoldi (one factorization, hundreds of solves on it).
        {"name": "eigen_tm_512_fp64", "kind": "eigen", "nx": 512, "ny": 512, "npml": 20,
         "pol": "TM", "precision": "fp64"},
        # A modulated guide: three sidebands, coupled solve, host arrays.
        {"name": "modulated_500x200_mixed", "kind": "modulated", "nx": 500, "ny": 200, "npml": 15,
         "pol": "TM", "precision": "mixed"},
        # A wavelength sweep with many sources in one batched call; one
        # source's fields are read back at every wavelength.
        {"name": "sweep_256_16x16_mixed", "kind": "sweep", "nx": 256, "ny": 256, "npml": 20,
         "pol": "TM", "precision": "mixed", "nomega": 16, "nsrc": 16},
        # Many sources on a factor that the program keeps (a scattering
        # matrix, a dipole scan), resident on the GPU.
        {"name": "sources_384x512_16_mixed", "kind": "sources", "nx": 384, "ny": 512, "npml": 20,
         "pol": "TM", "precision": "mixed", "nsrc": 16},
        # Guide modes for mode sources: 64 slices in one call.
        {"name": "modes_51x64", "kind": "modes", "n": 51, "count": 64, "pol": "TM"},
    ]


def draw(rng):
    """Sizes are log-uniform over the range of each kind, so odd and ragged
    ones occur; no drawn grid is larger than the largest listed one of its kind."""
    kind = rng.choice(["solve", "solve", "drive", "drive", "drive", "drive", "gradient", "eigen",
                       "modulated", "sweep", "sources", "sources", "modes"])

    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    if kind == "modes":
        return {"kind": kind, "n": size(31, 151), "count": size(4, 64),
                "pol": rng.choice(["TM", "TE"])}
    lo, hi = {"solve": (60, 300), "drive": (120, 1024), "gradient": (150, 700),
              "eigen": (100, 400), "modulated": (100, 300), "sweep": (64, 256),
              "sources": (100, 512)}[kind]
    c = {"kind": kind, "nx": size(lo, hi), "ny": size(lo, hi), "npml": rng.randint(8, 20),
         "pol": "TM" if kind in ("gradient", "modulated") else rng.choice(["TM", "TE"]),
         "precision": rng.choice(["mixed", "fp64"])}
    if kind == "sweep":
        c["nomega"], c["nsrc"] = size(2, 16), size(1, 16)
    if kind == "sources":
        c["nsrc"] = rng.choice([1, 1, 3, 8, 16])
    return c


# ---------------------------------------------------------------------------
# structures
# ---------------------------------------------------------------------------
def _omega(lam_um):
    return 2 * math.pi * core.C0 / (lam_um * 1e-6)


def _grid(c):
    lx, ly = c["nx"] * DL, c["ny"] * DL
    g = core.Grid(DL, (c["npml"], c["npml"]), (-lx / 2, lx / 2), (-ly / 2, ly / 2))
    assert g.N == (c["nx"], c["ny"])
    return g


def _pol(c):
    return core.TM if c["pol"] == "TM" else core.TE


def _coupler(c, seed):
    """Pixel design between two guides, and a short line source at the input."""
    nx, ny, npml = c["nx"], c["ny"], c["npml"]
    rng = np.random.default_rng([seed, nx, ny])
    eps = np.ones((nx, ny), dtype=np.complex128)
    side = max(1, int(round(600 / 1024 * min(nx, ny) / 8)))
    d = 8 * side
    x0, y0 = (nx - d) // 2, (ny - d) // 2
    yg = ny // 2 - 7
    eps[:x0, yg:yg + 15] = 12.25
    eps[x0 + d:, yg:yg + 15] = 12.25
    if c["kind"] == "gradient":  # a continuous design
        eps[x0:x0 + d, y0:y0 + d] = rng.uniform(1.0, 12.25, (d, d))
    else:
        pix = np.where(rng.random((side, side)) < 0.5, 12.25, 1.0)
        eps[x0:x0 + d, y0:y0 + d] = np.kron(pix, np.ones((8, 8)))
    src = np.zeros((nx, ny), dtype=np.complex128)
    ix = npml + 6 + int(rng.integers(0, 4))
    src[ix, ny // 2 - 12:ny // 2 + 13] = 1.0 + 0.2 * rng.standard_normal(25)
    return eps, src


def _points(c, seed):
    rng = np.random.default_rng([seed, 7, c["nx"], c["ny"]])
    s = np.zeros((c["nx"], c["ny"], c["nsrc"]), dtype=np.complex128)
    lo = c["npml"] + 1
    for r in range(c["nsrc"]):
        s[rng.integers(lo, max(lo + 1, c["nx"] // 4)), rng.integers(lo, c["ny"] - lo), r] = 1j
    return s


def _lattice(c, seed):
    """Triangular lattice of rods with one rod missing and rod permittivities
    that vary a little."""
    g = _grid(c)
    rng = np.random.default_rng([seed, 5, c["nx"], c["ny"]])
    a, r = 0.5, 0.1
    x, y = g.xc()[:, None], g.yc()[None, :]
    hx, hy = g.L[0] / 2, g.L[1] / 2
    eps = np.ones(g.N, dtype=np.complex128)
    for j in range(-int(hy / (a * math.sqrt(3) / 2)) - 1, int(hy / (a * math.sqrt(3) / 2)) + 2):
        y0 = a * j * math.sqrt(3) / 2
        n = int(hx / a + abs(j) / 2) + 2
        for i in range(-n, n + 1):
            x0 = a * (i + j / 2)
            if (i == 0 and j == 0) or abs(x0) > hx + r or abs(y0) > hy + r:
                continue
            ia, ib = np.searchsorted(x[:, 0], [x0 - r, x0 + r])
            ja, jb = np.searchsorted(y[0], [y0 - r, y0 + r])
            sub = eps[ia:ib + 1, ja:jb + 1]
            hit = (x[ia:ib + 1] - x0) ** 2 + (y[:, ja:jb + 1] - y0) ** 2 <= r * r
            sub[hit] = 8.9 + 0.2 * rng.standard_normal()
    return eps


def _modulated(c, seed):
    """A straight guide with a travelling modulation over its middle half."""
    rng = np.random.default_rng([seed, 11])
    nx, ny = c["nx"], c["ny"]
    eps = np.ones((nx, ny), dtype=np.complex128)
    deps = np.zeros((nx, ny), dtype=np.complex128)
    yg = ny // 2 - 5
    eps[:, yg:yg + 11] = 12.25
    k = rng.uniform(1.5, 2.5)
    x = np.arange(nx // 4, 3 * nx // 4)
    deps[x, yg:yg + 5] = (0.5 * np.exp(1j * k * DL * x))[:, None]
    src = np.zeros((nx, ny), dtype=np.complex128)
    src[c["npml"] + 10, yg - 3:yg + 14] = rng.uniform(0.5, 1.5, 17)
    return eps, deps, src


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------
def _device(a):
    """A host array Nx x Ny [x nsrc] as a device tensor in the library's layout."""
    a = a[:, :, None] if a.ndim == 2 else a
    flat = np.stack([a[:, :, r].ravel(order="F") for r in range(a.shape[2])])
    return torch.from_numpy(flat).cuda()


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def prepare(case, seed):
    logging.getLogger("fdfd").setLevel(logging.WARNING)
    c, kind = dict(case), case["kind"]
    s = {"case": c, "pol": _pol(c), "precision": c.get("precision")}
    if kind == "modes":
        rng = np.random.default_rng([seed, 3])
        n, m = c["n"], c["count"]
        eps = np.ones((m, n), dtype=np.complex128)
        eps[:, n // 2 - 7:n // 2 + 8] = 12.25 + 0.1 * rng.standard_normal((m, 1))
        s["slices"] = list(eps)
        s["omega"] = [_omega(lam) for lam in np.linspace(1.50, 1.60, m)]
        return s
    s["grid"] = _grid(c)
    om = _omega(1.55)
    if kind == "eigen":
        s["eps"] = _lattice(c, seed)
        s["omega"] = om
    elif kind == "modulated":
        eps, deps, src = _modulated(c, seed)
        s["device"] = modulated.ModulatedDevice(s["grid"], om, 2 * math.pi * 1e9, 1, eps_r=eps,
                                                deps_r=deps, src=src)
    elif kind == "sweep":
        eps, _ = _coupler(c, seed)
        s["eps"], s["srcs"] = eps, _points(c, seed)
        s["omega"] = [_omega(lam) for lam in np.linspace(1.50, 1.60, c["nomega"])]
    elif kind == "sources":
        # the program's own engine, holding the factor
        eps, _ = _coupler(c, seed)
        s["engine"] = Engine(0)
        s["engine"].set_grid(s["grid"])
        s["engine"].set_eps(eps)
        s["factor"], _ = s["engine"].factor(s["pol"], om, c["precision"])
        s["src"] = _device(_points(c, seed))
        s["out"] = torch.empty((c["nsrc"], 3, len(s["grid"])), dtype=torch.complex128, device="cuda")
    else:
        eps, src = _coupler(c, seed)
        if kind == "drive":
            s["omega"] = om
            s["eps"], s["src"] = _device(eps), _device(src)
            s["out"] = torch.empty((3, len(s["grid"])), dtype=torch.complex128, device="cuda")
        else:
            s["device"] = core.Device(s["grid"], om, eps, src)
            if kind == "gradient":  # mode overlap on a column before the right absorber
                m = np.zeros(s["grid"].N)
                y = (np.arange(c["ny"]) - c["ny"] // 2) * DL
                m[c["nx"] - c["npml"] - 8, :] = np.exp(-(y / 0.25) ** 2)
                s["overlap"] = m
    return s


def run(s):
    c, kind = s["case"], s["case"]["kind"]
    if kind == "solve":
        return fdfd.solve(s["device"], s["pol"], precision=s["precision"], tol=TOL).data
    if kind == "drive":
        eng = fdfd.engine()
        eng.set_grid(s["grid"])
        eng._chk(eng.lib.fdfd_set_eps_d(eng.h, _ptr(s["eps"])))
        fid, _ = eng.factor(s["pol"], s["omega"], s["precision"])
        st = _lib.fdfd_stats()
        eng._chk(eng.lib.fdfd_solve_d(eng.h, fid, 1, _ptr(s["src"]), _ptr(s["out"]), TOL, C.byref(st)))
        eng.release(fid)
        return s["out"]
    if kind == "gradient":
        j, grad, f = adjoint.objective_and_gradient(s["device"], s["overlap"],
                                                    precision=s["precision"], tol=TOL)
        return {"objective": j, "gradient": grad, "field": f.data}
    if kind == "eigen":
        eng = fdfd.engine()
        eng.set_grid(s["grid"])
        eng.set_eps(s["eps"])
        w, _, _ = eng.eigenfrequency(s["pol"], s["omega"], 8, ncv=20, precision=s["precision"],
                                     tol=TOL, want_fields=False)
        return w
    if kind == "modulated":
        fields = modulated.solve_modulated(s["device"], precision=s["precision"], tol=TOL)
        return [f.data for f in fields[0]]
    if kind == "sweep":
        job = (s["grid"], s["pol"], s["eps"], s["omega"], s["srcs"])
        got, _ = fdfd.engine().batch_solve([job], precision=s["precision"], tol=TOL,
                                           fetch=[(0, o, o % c["nsrc"]) for o in range(c["nomega"])])
        return [got[(0, o, o % c["nsrc"])] for o in range(c["nomega"])]
    if kind == "sources":
        eng, st = s["engine"], _lib.fdfd_stats()
        eng._chk(eng.lib.fdfd_solve_d(eng.h, s["factor"], c["nsrc"], _ptr(s["src"]), _ptr(s["out"]),
                                      TOL, C.byref(st)))
        return s["out"]
    beta, vecs, _ = modes.eigenmode_batch(s["slices"], DL, s["pol"], s["omega"], 3.0, 1)
    return {"beta": beta, "vectors": np.stack(vecs)}


# ---------------------------------------------------------------------------
# work and exact outputs
# ---------------------------------------------------------------------------
def work(case):
    """Inputs read once and outputs written once (16 bytes a complex value).
    Flops: a sparse direct factorization of a two-dimensional grid of N cells
    takes of the order of 10 N^1.5 complex multiply-adds under the best known
    ordering (nested dissection) and its triangular solves 16 N log2(N), at 8
    flops each; a mode slice takes 20 solves of a tridiagonal system."""
    kind = case["kind"]
    if kind == "modes":
        n, m = case["n"], case["count"]
        return {"bytes": 16.0 * m * (2 * n + 1), "flops": m * 20 * 8.0 * 20 * n}
    N = case["nx"] * case["ny"]
    factor = 8 * 10.0 * N ** 1.5
    solve = 8 * 16.0 * N * math.log2(N)
    field = 48.0 * N
    if kind in ("solve", "drive"):
        return {"bytes": 32.0 * N + field, "flops": factor + solve}
    if kind == "gradient":
        return {"bytes": 40.0 * N + field + 8.0 * N, "flops": factor + 2 * solve}
    if kind == "eigen":
        return {"bytes": 16.0 * N, "flops": factor + 60 * solve}
    if kind == "modulated":
        return {"bytes": 48.0 * N + 3 * field, "flops": 3 * factor + 9 * solve}
    if kind == "sweep":
        no, ns = case["nomega"], case["nsrc"]
        return {"bytes": 16.0 * N * (1 + ns) + no * ns * field, "flops": no * (factor + ns * solve)}
    return {"bytes": case["nsrc"] * (16.0 * N + field), "flops": case["nsrc"] * solve}


def _stretch(n, npml, omega):
    """1/s of the absorber on the forward and backward half-cells of one axis."""
    f, b = np.zeros(n), np.zeros(n)
    i = np.arange(npml)
    f[:npml], b[:npml] = npml - i - 0.5, npml - i
    f[n - npml:], b[n - npml:] = i + 0.5, i
    top = (3.5 + 1) * 12 / (2 * core.ETA0 * npml * DL)
    return tuple(1 / (1 - 1j * top * (d / npml) ** 3.5 / (omega * EPS0N)) for d in (f, b))


def _system(c, eps, omega):
    """The operator of one frequency, and the two maps from the solved
    component to the recovered ones."""
    import scipy.sparse as sp
    nx, ny = c["nx"], c["ny"]
    sxf, sxb = _stretch(nx, c["npml"], omega)
    syf, syb = _stretch(ny, c["npml"], omega)

    def diff(n):
        up = sp.diags([1.0], [1], shape=(n, n), format="lil")
        up[n - 1, 0] = 1.0
        return (up.tocsr() - sp.identity(n)) / DL

    fx, fy = diff(nx), diff(ny)
    ix, iy = sp.identity(nx), sp.identity(ny)
    dxf, dxb = sp.kron(iy, sp.diags(sxf) @ fx), sp.kron(iy, sp.diags(sxb) @ -fx.T)
    dyf, dyb = sp.kron(sp.diags(syf) @ fy, ix), sp.kron(sp.diags(syb) @ -fy.T, ix)
    e = EPS0N * eps
    if _pol(c) == core.TM:
        A = (dxf @ dxb + dyf @ dyb) / MU0N + omega ** 2 * sp.diags(e.ravel(order="F"))
        return A.tocsc(), -dyb / (1j * omega * MU0N), dxb / (1j * omega * MU0N)
    ex = sp.diags((2 / (e + np.roll(e, 1, axis=0))).ravel(order="F"))
    ey = sp.diags((2 / (e + np.roll(e, 1, axis=1))).ravel(order="F"))
    A = dxf @ ex @ dxb + dyf @ ey @ dyb + omega ** 2 * MU0N * sp.identity(nx * ny)
    return A.tocsc(), ey @ dyb / (1j * omega), -(ex @ dxb) / (1j * omega)


def _solved(system, omega, srcs):
    """All three components for each column of srcs, refined to rounding."""
    import scipy.sparse.linalg as sla
    A, m1, m2 = system
    lu = sla.splu(A, permc_spec="COLAMD")
    out = []
    for src in srcs:
        b = 1j * omega * src.ravel(order="F")
        x = lu.solve(b)
        for _ in range(3):
            x = x + lu.solve(b - A @ x)
        out.append(np.stack([x, m1 @ x, m2 @ x]))
    return out


def exact(case, seed):
    """scipy's sparse LU with refinement, where it takes seconds; mode slices
    by a dense eigenvalue solve."""
    c, kind = dict(case), case["kind"]
    if kind == "modes":
        return _modes_exact(c, seed)
    N = c["nx"] * c["ny"]
    if N > 210_000 or kind in ("gradient", "eigen", "modulated"):
        return None
    om = _omega(1.55)

    def whole(f):  # component-major vectors as Nx x Ny x 3
        return f.reshape(3, c["ny"], c["nx"]).transpose(2, 1, 0)

    eps, src = _coupler(c, seed)
    if kind == "solve":
        return whole(_solved(_system(c, eps, om), om, [src])[0])
    if kind == "drive":
        return _solved(_system(c, eps, om), om, [src])[0]
    p = _points(c, seed)
    if kind == "sources":
        return np.stack(_solved(_system(c, eps, om), om, [p[:, :, r] for r in range(c["nsrc"])]))
    out = [None] * c["nomega"]  # a sweep: its first, middle and last wavelength
    for o in sorted({0, c["nomega"] // 2, c["nomega"] - 1}):
        w = _omega(np.linspace(1.50, 1.60, c["nomega"])[o])
        out[o] = whole(_solved(_system(c, eps, w), w, [p[:, :, o % c["nsrc"]]])[0])
    return out


def _modes_exact(c, seed):
    """beta of the eigenvalue nearest (3 omega/c0)^2 of every slice, densely
    (the vectors' phase is left to the solver)."""
    s = prepare(c, seed)
    n = c["n"]
    beta = []
    for eps, om in zip(s["slices"], s["omega"]):
        f = (np.roll(np.eye(n), 1, axis=1) - np.eye(n)) / DL
        b = -f.T
        if s["pol"] == core.TM:
            A = om ** 2 * MU0N * EPS0N * np.diag(eps) + f @ b
        else:
            A = (om ** 2 * MU0N * EPS0N * np.diag(eps) +
                 np.diag(eps) @ f @ np.diag(2 / (eps + np.roll(eps, 1))) @ b)
        w = np.linalg.eigvals(A)
        k = int(np.argmin(np.abs(w - (3 * om * math.sqrt(MU0N * EPS0N)) ** 2)))
        beta.append([np.sqrt(w[k] + 0j)])
    return {"beta": np.array(beta), "vectors": None}
