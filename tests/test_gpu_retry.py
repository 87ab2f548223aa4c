"""What happens when the refinement on a dissected factor fails: an injected cut
is a failure by its residual, not by decree.  Grids and tolerances are those of
the error-path tests (96 x 80 cells, 1e-12)."""
import re

import numpy as np
import pytest

import fdfd_oracle as O
from fdfd import core
from fdfd._lib import FDFD_INJECT_NOCONV, FDFDError
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
