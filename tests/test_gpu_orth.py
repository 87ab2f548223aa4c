"""Orthogonalisation on the device: Arnoldi bases on both sides of the widths
its kernels are compiled for (2, 8, 32 vectors) and of what one launch takes
(32), and the lockstep solves of several sources on factors by lines, whose
bases grow to four vectors.

Eigenvalues agree with ARPACK's to 1e-9 relative: both are converged to 1e-12 in
theta = 1 / (lambda - sigma), and these few lie within a decade of the shift.
Solutions with a residual of 1e-12 agree to 1e-9 at the conditioning of these
grids (1e2 .. 1e3)."""
import numpy as np
import pytest

import fdfd_oracle as O
from fdfd import core
from fdfd.solve import Engine

pytestmark = pytest.mark.gpu


def _set(e, d):
    g = d.grid
    e.set_grid(core.Grid(g.dx, g.Npml, (g.bounds[0][0], g.bounds[1][0]),
                         (g.bounds[0][1], g.bounds[1][1]), g.L0))
    e.set_eps(d.eps_r)


@pytest.mark.parametrize("ncv", [8, 9, 31, 32, 33, 40])
def test_arnoldi_basis_widths(ncv):
    g = O.Grid.create(0.05, (5, 5), (0, 44 * 0.05), (0, 40 * 0.05))
    d = O.Device(g, O.omega_of_wavelength(1.6))
    d.eps_r[14:30, 12:28] = 9.0
    ref = O.eigenfrequency(d, O.TM, 3, tol=1e-14)[0]
    e = Engine(0)
    try:
        _set(e, d)
        om, _, st = e.eigenfrequency(O.TM, float(d.omega[0]), 3, ncv=ncv, tol=1e-12, want_fields=False)
        print(f"ncv={ncv}: {om} ref {ref} restarts={st['restarts']}", flush=True)
        assert st["nconv"] >= 3
        for w in om:
            assert np.min(np.abs(ref - w)) <= 1e-9 * abs(w)
    finally:
        e.close()


@pytest.mark.parametrize("nsrc", [2, 5, 16, 17])
@pytest.mark.parametrize("method", ["nd", "bcr"])
def test_lockstep_sources(monkeypatch, method, nsrc):
    if method == "bcr":
        monkeypatch.setenv("FDFD_METHOD", "bcr")
    g = O.Grid.create(0.03, (6, 5), (0, 61 * 0.03), (0, 48 * 0.03))
    d = O.Device(g, O.omega_of_wavelength(1.55))
    rng = np.random.default_rng(nsrc)
    d.eps_r[:] = 1 + 8 * rng.random(d.eps_r.shape)
    src = rng.standard_normal((61, 48, nsrc)) + 1j * rng.standard_normal((61, 48, nsrc))
    src[:, :, 1] = 0  # a source without a right-hand side keeps its place
    om = float(d.omega[0])
    A = O.assemble(g, d.eps_r, om, O.TM)
    e = Engine(0)
    try:
        _set(e, d)
        fid, _ = e.factor(O.TM, om, "mixed")
        f, st = e.solve_fields(fid, src, tol=1e-12)
        for r in range(nsrc):
            x = f[:, :, 0, r].ravel(order="F")
            b = O.rhs(om, src[:, :, r])
            if r == 1:
                assert not x.any()
                continue
            res = np.linalg.norm(b - A @ x) / np.linalg.norm(b)
            one, _ = e.linsolve(fid, b, tol=1e-12)
            err = np.linalg.norm(x - one) / np.linalg.norm(one)
            print(f"{method} source {r}/{nsrc}: res={res:.1e} against alone {err:.1e}", flush=True)
            assert res <= 1e-11 and err <= 1e-9
        assert st["iterations"] > nsrc if method == "bcr" else True
    finally:
        e.close()
