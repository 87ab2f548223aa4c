"""Negative permittivities on dissected factors, which do not pivot beyond blocks
of four cells: metal regions, and metal scattered at random so that every
separator and leaf holds some.  Solutions against the oracle's refined sparse LU at
the tolerances of the other solve tests (residual 1e-12, field 1e-10)."""
import numpy as np
import pytest

import fdfd_oracle as O
from fdfd import core
from fdfd.solve import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pol", [O.TM, O.TE])
@pytest.mark.parametrize("kind", ["block", "scattered"])
@pytest.mark.parametrize("Nx,Ny", [(44, 52), (150, 121)])
def test_metals(Nx, Ny, kind, pol):
    rng = np.random.default_rng(Nx)
    g = O.Grid.create(0.02, (6, 6), (0.0, Nx * 0.02), (0.0, Ny * 0.02))
    d = O.Device(g, O.omega_of_wavelength(1.55))
    if kind == "block":
        d.eps_r[Nx // 3:Nx // 2, Ny // 4:3 * Ny // 4] = -90 + 3j
    else:
        d.eps_r[:] = np.where(rng.random(g.N) < 0.3, -30 + 1j, 2.0)
    d.src[8:12, Ny // 2] = 1.0
    om = float(d.omega[0])
    ref = O.solve(d, pol)
    e = Engine(0)
    try:
        e.set_grid(core.Grid(g.dx, g.Npml, (g.bounds[0][0], g.bounds[1][0]),
                             (g.bounds[0][1], g.bounds[1][1]), g.L0))
        e.set_eps(d.eps_r)
        fid, fst = e.factor(pol, om, "fp64")
        f, st = e.solve_fields(fid, d.src, tol=1e-12)
        err = np.linalg.norm(f[:, :, :, 0] - ref.data) / np.linalg.norm(ref.data)
        print(f"{Nx}x{Ny} {kind} pol={pol}: err={err:.1e} its={st['iterations']}", flush=True)
        assert fst["pivot_fallback"] == 0 and st["residual"] <= 1e-12 and err <= 1e-10
    finally:
        e.close()
