"""fdfd_pack against numpy's transposition, exactly: every axis order, slices
with steps and negative strides, shapes around its tiles (8 and 32 cells, 16
sources), and arrays that the Python layer leaves to numpy (small ones, ones in
order, real ones, odd strides)."""
import itertools

import numpy as np
import pytest

from fdfd.solve import _flat, _pack


def _ref(a):
    return np.ascontiguousarray(np.asarray(a, dtype=np.complex128).transpose(2, 1, 0))


@pytest.mark.parametrize("shape", [(64, 65, 1), (33, 127, 1), (1, 4100, 1), (4100, 1, 1), (31, 9, 16), (40, 17, 17),
                                   (129, 95, 3), (700, 301, 1), (200, 130, 33)])
def test_every_axis_order(shape):
    rng = np.random.default_rng(shape[0])
    for order in itertools.permutations(range(3)):
        base = rng.standard_normal([shape[i] for i in order] + [2]).view(np.complex128)[..., 0]
        a = base.transpose(np.argsort(order))
        assert a.shape == shape
        got = _pack(a)
        assert got.flags.c_contiguous and np.array_equal(got, _ref(a))
        if shape[2] == 1:
            assert np.array_equal(_flat(a[:, :, 0]), _ref(a).ravel())


@pytest.mark.parametrize("sel", [np.s_[::2, :, :], np.s_[::-1, :, :], np.s_[:, ::-3, :], np.s_[3:, 5:, ::2]])
def test_slices(sel):
    rng = np.random.default_rng(7)
    a = (rng.standard_normal((150, 160, 4)) + 1j * rng.standard_normal((150, 160, 4)))[sel]
    assert np.array_equal(_pack(a), _ref(a))


def test_other_types_and_strides():
    rng = np.random.default_rng(8)
    r = rng.standard_normal((120, 90))
    assert np.array_equal(_flat(r), r.ravel(order="F").astype(complex))
    rec = np.zeros((120, 90), dtype=[("z", np.complex128), ("k", np.float64)])
    rec["z"] = r * (1 + 2j)
    assert np.array_equal(_flat(rec["z"]), rec["z"].ravel(order="F"))
    f = np.asfortranarray(r + 0j)
    assert np.shares_memory(_flat(f), f)  # in order already: no copy
    assert np.array_equal(_flat(np.arange(5.0)), np.arange(5) + 0j)
    four = (rng.standard_normal((40, 30, 5, 1)) + 0j)
    assert np.array_equal(_pack(four), _ref(four[..., 0]).reshape(5, -1))
