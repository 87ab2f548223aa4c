"""fdfd_autotune on grids that are dissected and on a handle that reduces lines:
the step time it reports is that of the steps that follow, and the variants that
it records are those that line factors are built with."""
import numpy as np
import pytest

import fdfd_oracle as O
from fdfd import core
from fdfd.solve import Engine

pytestmark = pytest.mark.gpu

P_ZBUILD = 5  # fdfd_profile_read: a kernel that only the line reduction launches


def _set(e, d):
    g = d.grid
    e.set_grid(core.Grid(g.dx, g.Npml, (g.bounds[0][0], g.bounds[1][0]),
                         (g.bounds[0][1], g.bounds[1][1]), g.L0))
    e.set_eps(d.eps_r)


@pytest.mark.parametrize("method", ["nd", "bcr"])
def test_reported_step_is_the_steps_that_follow(monkeypatch, method):
    """The device time of the better of three steps is the reported wall time less
    what the host adds (under 2 ms a step; the line reduction takes eleven times as
    long as the dissection here)."""
    if method == "bcr":
        monkeypatch.setenv("FDFD_METHOD", "bcr")
    else:
        monkeypatch.delenv("FDFD_METHOD", raising=False)
    d = O.random_pixel_device(512, 400, 16, 1.55, 3)
    om = float(d.omega[0])
    e = Engine(0)
    try:
        _set(e, d)
        _, ms = e.autotune(O.TM, om, "fp64")
        steps = []
        for _ in range(3):
            fid, fst = e.factor(O.TM, om, "fp64")
            _, st = e.solve_fields(fid, d.src, tol=1e-10)
            e.release(fid)
            steps.append(fst["t_factor_ms"] + st["t_solve_ms"])
        print(f"{method}: reported {ms:.2f} ms, device {min(steps):.2f} ms", flush=True)
        assert 0.7 * min(steps) <= ms <= 1.5 * min(steps) + 2.0
    finally:
        e.close()


@pytest.mark.parametrize("precision", ["mixed", "fp64"])
def test_recorded_variants_build_line_factors(monkeypatch, tmp_path, precision):
    monkeypatch.setenv("FDFD_METHOD", "bcr")
    monkeypatch.setenv("FDFD_TUNE_CACHE", str(tmp_path / "tune.txt"))
    d = O.random_pixel_device(128, 96, 10, 1.55, 21)
    om = float(d.omega[0])
    e1, e2 = Engine(0), Engine(0)
    try:
        _set(e1, d)
        knobs, _ = e1.autotune(O.TM, om, precision)
        _set(e2, d)
        e2.profile()
        fid, _ = e2.factor(O.TM, om, precision)
        assert e2.tuning() == knobs and e2.profile_read(P_ZBUILD)["launches"] > 0
        e2.profile(False)
        f, _ = e2.solve_fields(fid, d.src, tol=1e-12)
        ref = O.solve(d, O.TM)
        assert np.linalg.norm(f[:, :, :, 0] - ref.data) <= 1e-10 * np.linalg.norm(ref.data)
    finally:
        e1.close()
        e2.close()
