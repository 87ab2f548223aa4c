"""Nested-dissection factors against the line reduction (FDFD_METHOD=bcr) and
the oracle's matrix, on grids where the tree changes shape: the smallest the
dissection takes (min(Nx, Ny) = 16), leaves of one and several sizes, ragged
and elongated grids cut along either side, separators on both sides of the
32-cell panel and 64-cell window, and one level with Q and Schur products on
the large tiles.  Both factors precondition the same FGMRES, so the solutions
agree to the requested residual times the conditioning (1e-10 at 1e-13)."""
import numpy as np
import pytest

import fdfd_oracle as O
from fdfd import core
from fdfd.solve import Engine

pytestmark = pytest.mark.gpu


def _device(Nx, Ny, npml, seed):
    rng = np.random.default_rng(seed)
    g = O.Grid.create(0.02, (npml, npml), (0.0, Nx * 0.02), (0.0, Ny * 0.02))
    d = O.Device(g, O.omega_of_wavelength(1.55))
    d.eps_r[:] = 1 + 11.25 * rng.random((Nx, Ny)) + 0.1j * rng.random((Nx, Ny))
    d.src[:] = rng.standard_normal((Nx, Ny)) + 1j * rng.standard_normal((Nx, Ny))
    return d


def _engine(monkeypatch, method, d):
    if method == "bcr":
        monkeypatch.setenv("FDFD_METHOD", "bcr")
    else:
        monkeypatch.delenv("FDFD_METHOD", raising=False)
    e = Engine(0)
    g = d.grid
    e.set_grid(core.Grid(0.02, g.Npml, (g.bounds[0][0], g.bounds[1][0]),
                         (g.bounds[0][1], g.bounds[1][1]), g.L0))
    e.set_eps(d.eps_r)
    return e


@pytest.mark.parametrize("pol", [O.TM, O.TE])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("Nx,Ny,npml", [(16, 16, 0), (16, 61, 3), (17, 40, 2), (33, 16, 4), (64, 65, 6),
                                        (129, 70, 8), (31, 500, 6), (300, 270, 9)])
def test_dissection_matches_line_reduction(monkeypatch, Nx, Ny, npml, precision, pol):
    d = _device(Nx, Ny, npml, 100 * Nx + Ny)
    om = float(d.omega[0])
    A = O.assemble(d.grid, d.eps_r, om, pol)
    b = O.rhs(om, d.src)
    x = {}
    for method in ("nd", "bcr"):
        e = _engine(monkeypatch, method, d)
        try:
            fid, fst = e.factor(pol, om, precision)
            for tr in (False, True):
                y, st = e.linsolve(fid, b, transpose=tr, tol=1e-13)
                res = np.linalg.norm(b - (A.T if tr else A) @ y) / np.linalg.norm(b)
                print(f"{method} {Nx}x{Ny} pol={pol} {precision} tr={tr}: res={res:.1e} "
                      f"its={st['iterations']}", flush=True)
                assert res <= 1e-12
                x[method, tr] = y
            e.release(fid)
            assert fst["pivot_fallback"] == 0
        finally:
            e.close()
    for tr in (False, True):
        err = np.linalg.norm(x["nd", tr] - x["bcr", tr]) / np.linalg.norm(x["bcr", tr])
        assert err <= 1e-10


def test_several_grids_share_a_handle(monkeypatch):
    """More grid shapes than a handle keeps trees for, in turn and again."""
    e = Engine(0)
    try:
        for Nx, Ny in [(40, 30), (30, 40), (52, 24), (24, 52), (44, 44), (40, 30)]:
            d = _device(Nx, Ny, 4, Nx + Ny)
            g = d.grid
            e.set_grid(core.Grid(0.02, g.Npml, (g.bounds[0][0], g.bounds[1][0]),
                                 (g.bounds[0][1], g.bounds[1][1]), g.L0))
            e.set_eps(d.eps_r)
            om = float(d.omega[0])
            fid, _ = e.factor(O.TM, om, "mixed")
            x, _ = e.linsolve(fid, O.rhs(om, d.src), tol=1e-13)
            b = O.rhs(om, d.src)
            assert np.linalg.norm(b - O.assemble(g, d.eps_r, om, O.TM) @ x) <= 1e-12 * np.linalg.norm(b)
    finally:
        e.close()


@pytest.mark.parametrize("Nx,Ny", [(16, 16), (18, 18), (20, 20), (22, 22), (24, 24), (28, 28), (19, 30), (16, 27)])
def test_leaf_fronts_of_every_size(monkeypatch, Nx, Ny):
    """Leaves of 20 to 49 cells with boundaries of 16 to 32: the last swept block
    ends inside its 16-cell tile after 4, 8, 12 or 16 cells, with boundary rows
    behind it.  FP64 factors leave a relative residual near 1e-13 after one
    application, so a sound one needs at most two iterations for 1e-13 (a wrong
    entry costs many or never converges)."""
    d = _device(Nx, Ny, 2, Nx * 31 + Ny)
    om = float(d.omega[0])
    b = O.rhs(om, d.src)
    e = _engine(monkeypatch, "nd", d)
    try:
        for pol in (O.TM, O.TE):
            fid, fst = e.factor(pol, om, "fp64")
            x, st = e.linsolve(fid, b, tol=1e-13)
            res = np.linalg.norm(b - O.assemble(d.grid, d.eps_r, om, pol) @ x) / np.linalg.norm(b)
            print(f"{Nx}x{Ny} pol={pol}: res={res:.1e} its={st['iterations']}", flush=True)
            assert fst["pivot_fallback"] == 0 and st["iterations"] <= 2 and res <= 1e-12
            e.release(fid)
    finally:
        e.close()


@pytest.mark.parametrize("K", [3, 4])
def test_sideband_factors_side_by_side(K):
    """Seven and nine sideband factors: fewer and more than one launch takes
    (eight).  Same bar as the modulated solve's other tests, 1e-10 of the largest
    sideband at a residual of 1e-13."""
    from test_gpu_modulated import _check, _pair
    from fdfd.modulated import solve_modulated
    d, o = _pair(48, 40, 4, K, True, seed=20 + K)
    e = Engine(0)
    try:
        fg, st = solve_modulated(d, precision="fp64", tol=1e-13, eng=e, return_stats=True)
        assert st[0]["residual"] <= 1e-13
        _check(fg[0], O.solve_modulated(o)[0], f"K={K}")
    finally:
        e.close()


@pytest.mark.parametrize("Nx,Ny", [(17, 300), (17, 17), (26, 26), (32, 32), (34, 34), (36, 36), (100, 16)])
def test_small_fronts_whole(monkeypatch, Nx, Ny):
    """Levels of 4, 8, 12 and 16 separator cells with 16 to 84 boundary cells, on
    both sides of 64, where the kernel of whole fronts changes size; one child or
    two.  Same bar as the leaves'."""
    test_leaf_fronts_of_every_size(monkeypatch, Nx, Ny)


@pytest.mark.parametrize("Nx,Ny", [(66, 68), (128, 129), (132, 150), (193, 196), (257, 260)])
def test_long_separators(monkeypatch, Nx, Ny):
    """Separators swept in blocks of 64: two to five of them, the last one of 4
    cells, nearly or quite full.  Same bar as the leaves'."""
    test_leaf_fronts_of_every_size(monkeypatch, Nx, Ny)
