"""A batch looks its jobs' factor sizes up once for each grid shape: what it does
before any device work (sizes, order of the groups, release of the handle's
factors; the first line of FDFD_DEBUG_TIMING) does not grow with the jobs.  A
dissection tree of 960 x 960 cells takes a few tenths of a millisecond to build, and 64 jobs are
some 300 comparisons of a sort (0.07 s where each built two trees)."""
import re

import numpy as np
import pytest

import fdfd_oracle as O
from fdfd import core
from fdfd.solve import Engine

pytestmark = pytest.mark.gpu


def test_many_jobs_are_planned_once(monkeypatch, capfd):
    monkeypatch.delenv("FDFD_METHOD", raising=False)
    monkeypatch.setenv("FDFD_DEBUG_TIMING", "1")
    g = core.Grid(0.02, (12, 12), (0.0, 19.2), (0.0, 19.2))
    assert g.N == (960, 960)
    eps = np.full(g.N, 2.25 + 0j, order="F")
    src = np.zeros((960, 960, 1), dtype=complex, order="F")
    src[480, 480] = 1j
    om = [O.omega_of_wavelength(1.55)]
    before = {}
    e = Engine(0)
    try:
        for jobs in (1, 64):
            capfd.readouterr()
            res, st = e.batch_solve([(g, O.TM, eps, om, src)] * jobs, tol=1e-10,
                                    fetch=[(0, 0, 0), (jobs - 1, 0, 0)])
            err = capfd.readouterr().err
            before[jobs] = float(re.search(r"handle's factors and pool: ([0-9.]+) s", err).group(1))
            assert st["residual"] <= 1e-10
            assert np.array_equal(res[0, 0, 0], res[jobs - 1, 0, 0])
        print(before, flush=True)
        assert before[64] <= before[1] + 0.03
    finally:
        e.close()
