"""What happens when the refinement on a dissected factor fails: an injected cut
is a failure by its residual, not by decree; a factor that no refinement converges
on (FDFD_INJECT_POOR_FACTOR) is rebuilt by the line reduction and the solve
repeated, for one source, several, transposed, coupled sidebands and batches.
Grids and tolerances are those of the error-path tests (96 x 80 cells, residual
1e-12, fields 1e-10)."""
import ctypes as C
import re

import numpy as np
import pytest

import fdfd_oracle as O
from fdfd import core
from fdfd._lib import (FDFD_INJECT_NOCONV, FDFD_INJECT_OOM, FDFD_INJECT_PIVOT_FALLBACK,
                       FDFD_INJECT_POOR_FACTOR, FDFDError)
from fdfd.solve import Engine

pytestmark = pytest.mark.gpu


def _cgrid(g):
    return core.Grid(g.dx, g.Npml, (g.bounds[0][0], g.bounds[1][0]),
                     (g.bounds[0][1], g.bounds[1][1]), g.L0)


@pytest.fixture(scope="module")
def small():
    d = O.random_pixel_device(96, 80, 10, 1.55, 7)
    return d, float(d.omega[0]), O.solve(d, O.TM)


def _engine(monkeypatch, method, d):
    if method == "bcr":
        monkeypatch.setenv("FDFD_METHOD", "bcr")
    else:
        monkeypatch.delenv("FDFD_METHOD", raising=False)
    e = Engine(0)
    e.set_grid(_cgrid(d.grid))
    e.set_eps(d.eps_r)
    return e


def _residual(msg):
    return float(re.search(r"relative residual ([0-9.e+-]+|nan|inf)", msg).group(1))


@pytest.mark.parametrize("method", ["nd", "bcr"])
def test_cut_refinement_names_its_residual(monkeypatch, small, method):
    """One iteration on complex64 line factors, or on half of a dissected one, is
    too few for 1e-12, and the error says what was reached.  The factor is as it
    was: the next solve takes as many iterations as the one before."""
    d, om, ref = small
    e = _engine(monkeypatch, method, d)
    try:
        fid, _ = e.factor(O.TM, om, "mixed")
        _, before = e.solve_fields(fid, d.src, tol=1e-12)
        e.debug_inject(FDFD_INJECT_NOCONV, 1)
        with pytest.raises(FDFDError) as ei:
            e.solve_fields(fid, d.src, tol=1e-12)
        print(method, ei.value, flush=True)
        assert ei.value.code == -4 and 1e-12 < _residual(str(ei.value)) <= 1.0 + 1e-9
        f, st = e.solve_fields(fid, d.src, tol=1e-12)
        assert st["iterations"] == before["iterations"]
        assert np.linalg.norm(f[:, :, :, 0] - ref.data) <= 1e-10 * np.linalg.norm(ref.data)
    finally:
        e.close()


def test_cut_that_suffices_is_no_failure(monkeypatch, small):
    d, om, _ = small
    e = _engine(monkeypatch, "bcr", d)
    try:
        fid, _ = e.factor(O.TM, om, "mixed")
        e.debug_inject(FDFD_INJECT_NOCONV, 30)
        _, st = e.solve_fields(fid, d.src, tol=1e-12)
        assert st["residual"] <= 1e-12
    finally:
        e.close()


def _field_err(f, ref):
    return np.linalg.norm(f - ref) / np.linalg.norm(ref)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_poor_factor_is_rebuilt_for_one_source(monkeypatch, small, precision):
    d, om, ref = small
    e = _engine(monkeypatch, "nd", d)
    try:
        e.debug_inject(FDFD_INJECT_POOR_FACTOR)
        fid, fst = e.factor(O.TM, om, precision)
        f, st = e.solve_fields(fid, d.src, tol=1e-12)
        print(precision, st, flush=True)
        assert fst["pivot_fallback"] == 0 and st["pivot_fallback"] == 1
        assert st["residual"] <= 1e-12 and _field_err(f[:, :, :, 0], ref.data) <= 1e-10
        f, again = e.solve_fields(fid, d.src, tol=1e-12)  # on the rebuilt factor
        assert again["iterations"] < 30 and _field_err(f[:, :, :, 0], ref.data) <= 1e-10
        e.release(fid)
        fid, _ = e.factor(O.TM, om, precision)  # one-shot
        _, st = e.solve_fields(fid, d.src, tol=1e-12)
        assert st["pivot_fallback"] == 0
    finally:
        e.close()


def test_poor_factor_is_rebuilt_for_transposed_solves(monkeypatch, small):
    d, om, _ = small
    b = O.rhs(om, d.src)
    A = O.assemble(d.grid, d.eps_r, om, O.TM)
    e = _engine(monkeypatch, "nd", d)
    try:
        e.debug_inject(FDFD_INJECT_POOR_FACTOR)
        fid, _ = e.factor(O.TM, om, "fp64")
        x, st = e.linsolve(fid, b, transpose=True, tol=1e-12)
        assert st["pivot_fallback"] == 1
        assert np.linalg.norm(b - A.T @ x) <= 1e-11 * np.linalg.norm(b)
    finally:
        e.close()


def test_poor_factor_is_rebuilt_for_several_sources(monkeypatch, small):
    d, om, ref = small
    src = np.stack([d.src, np.zeros_like(d.src), np.roll(d.src, 7, axis=1)], axis=2)
    e = _engine(monkeypatch, "nd", d)
    try:
        e.debug_inject(FDFD_INJECT_POOR_FACTOR)
        fid, _ = e.factor(O.TM, om, "mixed")
        f, st = e.solve_fields(fid, src, tol=1e-12)
        assert st["pivot_fallback"] == 1 and st["residual"] <= 1e-12
        assert _field_err(f[:, :, :, 0], ref.data) <= 1e-10 and not f[:, :, :, 1].any()
        x, _ = O.linear_solve(O.assemble(d.grid, d.eps_r, om, O.TM), O.rhs(om, src[:, :, 2]))
        assert _field_err(f[:, :, 0, 2].ravel(order="F"), x) <= 1e-10
    finally:
        e.close()


@pytest.mark.parametrize("poor", [0, 1, 2])
def test_poor_sideband_factor_is_rebuilt(monkeypatch, poor):
    from test_gpu_modulated import _check, _pair
    from fdfd.modulated import solve_modulated
    monkeypatch.delenv("FDFD_METHOD", raising=False)
    d, o = _pair(48, 40, 4, 1, True, seed=11)
    e = Engine(0)
    try:
        e.debug_inject(FDFD_INJECT_POOR_FACTOR, poor)
        fg, st = solve_modulated(d, precision="fp64", tol=1e-13, eng=e, return_stats=True)
        assert st[0]["pivot_fallback"] == 1 and st[0]["residual"] <= 1e-13
        _check(fg[0], O.solve_modulated(o)[0], f"poor sideband {poor}")
    finally:
        e.close()


@pytest.mark.parametrize("poor", [0, 2])
def test_poor_factor_is_rebuilt_inside_a_batch(monkeypatch, poor):
    """Two jobs are two groups: the second is factored by the builder's thread
    while the first group's solve rebuilds its poor factor."""
    monkeypatch.delenv("FDFD_METHOD", raising=False)
    oms = np.array([O.omega_of_wavelength(l) for l in (1.50, 1.54, 1.58)])
    ds = [O.random_pixel_device(96, 80, 10, 1.55, 7), O.random_pixel_device(72, 88, 10, 1.55, 8)]
    e = Engine(0)
    try:
        e.debug_inject(FDFD_INJECT_POOR_FACTOR, poor)
        srcs = [np.stack([d.src, np.roll(d.src, 5, axis=1)], axis=2) for d in ds]
        res, st = e.batch_solve([(_cgrid(d.grid), O.TM, d.eps_r, oms, s) for d, s in zip(ds, srcs)],
                                precision="mixed", tol=1e-12)
        assert st["pivot_fallback"] == 1 and st["residual"] <= 1e-12
        for d, s, r in zip(ds, srcs, res):
            for o, w in enumerate(oms):
                A = O.assemble(d.grid, d.eps_r, float(w), O.TM)
                for k in range(2):
                    x, _ = O.linear_solve(A, O.rhs(float(w), s[:, :, k]))
                    assert _field_err(r[o, k, :, :, 0].ravel(order="F"), x) <= 1e-10, (o, k)
    finally:
        e.close()


@pytest.mark.parametrize("poor", [1, 2])
def test_poor_sideband_beside_a_line_factor(monkeypatch, poor):
    """Sideband 0 fails its pivot check and is a line factor from the start;
    another one is poor."""
    from test_gpu_modulated import _check, _pair
    from fdfd.modulated import solve_modulated
    monkeypatch.delenv("FDFD_METHOD", raising=False)
    d, o = _pair(48, 40, 4, 1, True, seed=11)
    e = Engine(0)
    try:
        e.debug_inject(FDFD_INJECT_PIVOT_FALLBACK)
        e.debug_inject(FDFD_INJECT_POOR_FACTOR, poor)
        fg, st = solve_modulated(d, precision="fp64", tol=1e-13, eng=e, return_stats=True)
        assert st[0]["residual"] <= 1e-13
        _check(fg[0], O.solve_modulated(o)[0], f"poor sideband {poor} beside a line factor")
    finally:
        e.close()


@pytest.mark.parametrize("nsrc", [1, 3])
def test_no_room_for_line_factors(monkeypatch, small, nsrc):
    """Where the line factor cannot be had, the solve has failed to converge and says
    so, with its residual; a later one, with memory back, rebuilds and succeeds."""
    d, om, ref = small
    src = np.stack([d.src] * nsrc, axis=2)
    e = _engine(monkeypatch, "nd", d)
    try:
        e.debug_inject(FDFD_INJECT_POOR_FACTOR)
        fid, _ = e.factor(O.TM, om, "fp64")
        e.debug_inject(FDFD_INJECT_OOM)
        with pytest.raises(FDFDError) as ei:
            e.solve_fields(fid, src, tol=1e-12)
        assert ei.value.code == -4 and _residual(str(ei.value)) > 1e-12
        f, st = e.solve_fields(fid, src, tol=1e-12)
        assert st["pivot_fallback"] == 1 and _field_err(f[:, :, :, 0], ref.data) <= 1e-10
    finally:
        e.close()


@pytest.mark.parametrize("pol", [O.TM, O.TE])
@pytest.mark.parametrize("tol", [1e-16, 1e-18])
@pytest.mark.parametrize("npml", [0, 10])
def test_tolerance_below_rounding_keeps_the_factor(monkeypatch, pol, tol, npml):
    """A residual of a few 1e-15 is what rounding leaves of any solve here, so lower
    tolerances fail (they did on line factors too) and the factor is not to blame:
    it stays, whether one source asked, several, or the transposed system."""
    d = O.random_pixel_device(96, 80, npml, 1.55, 7)
    om = float(d.omega[0])
    b = O.rhs(om, d.src) if npml else O.rhs(om, np.roll(d.src, 30, axis=0))
    src = b.reshape(d.grid.N, order="F") / (1j * om)
    e = _engine(monkeypatch, "nd", d)
    try:
        fid, _ = e.factor(pol, om, "fp64")
        calls = [lambda t: e.solve_fields(fid, src, tol=t)[1],
                 lambda t: e.solve_fields(fid, np.stack([src, np.roll(src, 3, axis=1)], axis=2), tol=t)[1],
                 lambda t: e.linsolve(fid, b, tol=t)[1],
                 lambda t: e.linsolve(fid, b, transpose=True, tol=t)[1]]
        for call in calls:
            with pytest.raises(FDFDError) as ei:
                call(tol)
            assert ei.value.code == -4 and _residual(str(ei.value)) <= 1e-11
            assert call(1e-10)["pivot_fallback"] == 0
    finally:
        e.close()


def test_tolerance_below_rounding_keeps_sideband_factors(monkeypatch):
    from test_gpu_modulated import _pair
    from fdfd.modulated import solve_modulated
    monkeypatch.delenv("FDFD_METHOD", raising=False)
    d, _ = _pair(48, 40, 4, 1, True, seed=11)
    e = Engine(0)
    rcs = []
    e._chk = rcs.append  # the statistics of the failed solve, in place of its error
    try:
        _, st = solve_modulated(d, precision="fp64", tol=1e-18, eng=e, return_stats=True)
        print(rcs, st, flush=True)
        assert rcs[-1] == -4 and 0 < st[0]["residual"] <= 1e-13 and st[0]["pivot_fallback"] == 0
    finally:
        e.close()


@pytest.mark.parametrize("nsrc", [1, 3])
def test_factor_that_is_not_finite_is_rebuilt(monkeypatch, small, nsrc):
    """Residuals that are not numbers end the refinement at once (it used to restart
    40 times on them) and the factor is rebuilt."""
    d, om, ref = small
    e = _engine(monkeypatch, "nd", d)
    try:
        e.debug_inject(FDFD_INJECT_POOR_FACTOR, -1)
        fid, _ = e.factor(O.TM, om, "fp64")
        f, st = e.solve_fields(fid, np.stack([d.src] * nsrc, axis=2), tol=1e-12)
        print(st, flush=True)
        assert st["pivot_fallback"] == 1 and st["iterations"] <= 5 * nsrc
        assert _field_err(f[:, :, :, nsrc - 1], ref.data) <= 1e-10
        e.debug_inject(FDFD_INJECT_POOR_FACTOR, -1)
        fid, _ = e.factor(O.TM, om, "fp64")
        b = O.rhs(om, d.src)
        x, st = e.linsolve(fid, b, transpose=True, tol=1e-12)
        A = O.assemble(d.grid, d.eps_r, om, O.TM)
        assert st["pivot_fallback"] == 1 and np.linalg.norm(b - A.T @ x) <= 1e-11 * np.linalg.norm(b)
    finally:
        e.close()


@pytest.mark.parametrize("nsrc", [1, 3])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_source_that_is_not_finite_keeps_the_factor(monkeypatch, small, nsrc, value):
    d, om, ref = small
    src = np.stack([d.src] * nsrc, axis=2)
    src[40, 40, 0] = value
    e = _engine(monkeypatch, "nd", d)
    chk, rcs = e._chk, []
    try:
        fid, _ = e.factor(O.TM, om, "fp64")
        e._chk = rcs.append  # the statistics of the failed solve, in place of its error
        _, st = e.solve_fields(fid, src, tol=1e-12)
        e._chk = chk
        assert rcs == [-4] and not np.isfinite(st["residual"]) and st["iterations"] <= 5 * nsrc
        f, st = e.solve_fields(fid, d.src, tol=1e-12)
        assert st["pivot_fallback"] == 0 and _field_err(f[:, :, :, 0], ref.data) <= 1e-10
    finally:
        e.close()


@pytest.mark.parametrize("cells", [2, 4])
@pytest.mark.parametrize("value", [1e70, 1e82, 1e120])
def test_pivots_out_of_range(monkeypatch, value, cells):
    """Permittivities that take the last pivot blocks out of the range their
    reciprocal works in (squares up to 1e308), with no later pivot to show it: the
    factor is one by lines, as it would have been without the dissection.  The
    cells are the last ones eliminated, on the column that cuts the torus."""
    d = O.random_pixel_device(96, 80, 10, 1.55, 7)
    d.eps_r[-1, -cells:] = value
    om = float(d.omega[0])
    b = O.rhs(om, d.src)
    b[np.real(d.eps_r.ravel(order="F")) > 1e50] = 0
    e = _engine(monkeypatch, "nd", d)
    try:
        fid, fst = e.factor(O.TM, om, "fp64")
        x, st = e.linsolve(fid, b, tol=1e-11)
        res = np.linalg.norm(b - O.assemble(d.grid, d.eps_r, om, O.TM) @ x) / np.linalg.norm(b)
        print(f"eps {value:.0e} in {cells} cells: fallback {fst['pivot_fallback']} its {st['iterations']} res {res:.1e}",
              flush=True)
        assert fst["pivot_fallback"] == (1 if value > 1e80 else 0) and res <= 1e-10
    finally:
        e.close()


def test_allocation_failure_leaves_no_error_behind(monkeypatch, small):
    """A batch whose results do not fit (10000 wavelengths at 1024 x 1024, 500 GB) is
    refused, and the next call does not report that again."""
    d, om, ref = small
    e = _engine(monkeypatch, "nd", d)
    g = core.Grid(0.02, (8, 8), (0.0, 1024 * 0.02), (0.0, 1024 * 0.02))
    try:
        with pytest.raises(FDFDError) as ei:
            e.batch_solve([(g, O.TM, np.ones(g.N), om * np.linspace(1, 1.1, 10000), np.ones(g.N))], keep=False)
        assert ei.value.code == -2
        e.set_grid(_cgrid(d.grid))
        e.set_eps(d.eps_r)
        fid, _ = e.factor(O.TM, om, "fp64")
        f, _ = e.solve_fields(fid, d.src, tol=1e-12)
        assert _field_err(f[:, :, :, 0], ref.data) <= 1e-10
    finally:
        e.close()


def test_work_that_does_not_fit_is_allocated_again(monkeypatch, small):
    """A factorization whose work does not fit (1024 lines of 700000 cells) frees the
    work of smaller ones; they get theirs anew."""
    d, om, ref = small
    e = _engine(monkeypatch, "bcr", d)
    hip = C.CDLL("libamdhip64.so")
    hip.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
    hip.hipFree.argtypes = [C.c_void_p]
    try:
        for again in (False, True):
            if again:
                g = core.Grid(0.02, (8, 8), (0.0, 1024 * 0.02), (0.0, 700000 * 0.02))
                e.set_grid(g)
                eps = C.c_void_p()  # (its values are not looked at)
                assert hip.hipMalloc(C.byref(eps), 16 * len(g)) == 0
                e._chk(e.lib.fdfd_set_eps_d(e.h, eps))
                assert hip.hipFree(eps) == 0
                with pytest.raises(FDFDError) as ei:
                    e.factor(O.TM, om, "fp64")
                assert ei.value.code == -2
                e.set_grid(_cgrid(d.grid))
                e.set_eps(d.eps_r)
            fid, _ = e.factor(O.TM, om, "fp64")
            f, _ = e.solve_fields(fid, d.src, tol=1e-12)
            assert _field_err(f[:, :, :, 0], ref.data) <= 1e-10
            e.release(fid)
    finally:
        e.close()
