"""1-D modes where the wave-wide recurrences and the projected eigenproblem
change shape: slices around 64-row chunks, the shortest ones, those on both
sides of the 1056 cells whose rows are formed in LDS, and bases from the
smallest to all 32 vectors, with restarts.

The Arnoldi residual is at most 1e-12 |theta| in (A - sigma)^-1, so
|A v - beta^2 v| <= 1e-12 |A - sigma| (with rounding, 1e-10 of the operator's
norm); where the dense spectrum is at hand the eigenvalues are its nearest to the
shift to 1e-9 relative to that norm."""
import numpy as np
import pytest

import fdfd_oracle as O
from fdfd import modes
from fdfd.solve import Engine

pytestmark = pytest.mark.gpu
OM = O.omega_of_wavelength(1.55)


def _check(e, n, pol, nev, ncv):
    rng = np.random.default_rng(n + 7 * ncv)
    eps = 2.25 + 0.1 * rng.random(n) + 0.01j
    eps[n // 3:n // 3 + max(1, n // 4)] = 12.25
    neff = 3.2
    A = O.mode_operator_1d(eps, 0.02, OM, pol)
    norm = abs(A).sum(axis=1).max()
    beta, vecs, st = modes.eigenmode_batch([eps, eps[::-1].copy()], 0.02, pol, OM, neff, nev, ncv=ncv, eng=e)
    lam, v = beta[0] ** 2, vecs[0]
    res = np.linalg.norm(A @ v - v * lam, axis=0).max() / norm
    print(f"n={n} pol={pol} nev={nev} ncv={ncv}: residual {res:.1e} restarts {st['restarts']}", flush=True)
    assert st["nconv"] >= nev and res <= 1e-10
    assert np.abs(np.linalg.norm(v, axis=0) - 1).max() <= 1e-12
    if n <= 200:
        _, _, c0 = O.normalize_parameters(O.DEFAULT_L0)
        sigma = (OM / c0 * neff) ** 2
        w = np.linalg.eigvals(A.toarray())
        near = np.sort(np.abs(w - sigma))[:nev]
        assert np.abs(np.sort(np.abs(lam - sigma)) - near).max() <= 1e-9 * norm


@pytest.fixture(scope="module")
def eng():
    e = Engine(0)
    yield e
    e.close()


@pytest.mark.parametrize("pol", [O.TM, O.TE])
@pytest.mark.parametrize("n", [3, 4, 5, 62, 63, 64, 65, 66, 67, 127, 128, 129, 130, 1056, 1057])
def test_slice_lengths(eng, n, pol):
    _check(eng, n, pol, 1, 0)


@pytest.mark.parametrize("nev,ncv", [(1, 3), (2, 5), (1, 31), (1, 32), (3, 9), (12, 32), (29, 32)])
def test_basis_sizes(eng, nev, ncv):
    _check(eng, 75, O.TM, nev, ncv)
