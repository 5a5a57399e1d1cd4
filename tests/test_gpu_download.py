"""Fields come back as they went in, at the edges of the download's chunks: a field of one
chunk and of several, odd and even row lengths (a pair of values may span two rows), both
device layouts, and leading dimensions larger than the field's."""
import ctypes

import numpy as np
import pytest

from pixelflow_amd import cases

pytestmark = pytest.mark.gpu


def _params(size):
    m, n, l = size
    return cases.CaseParams(dim=3 if l > 1 else 2, m=m, n=n, l=l, width=0.01 * (m - 1), height=0.01 * (n - 1),
                            depth=0.01 * (l - 1) if l > 1 else 0.0, time=1e-3, istep_max=10, iter_max=5)


@pytest.mark.parametrize("size", [(3, 3, 3), (5, 4, 1), (97, 51, 1), (130, 96, 90), (129, 95, 91), (1001, 1201, 1)])
def test_field_round_trip(size):
    from pixelflow_amd.solver import FIELDS, Solver, lib
    p = _params(size)
    shape = p.full_shape()
    rng = np.random.default_rng(sum(size))
    with Solver(p, np.ones(p.interior_shape())) as s:
        for f in ("u", "p"):
            a = rng.standard_normal(shape)
            s.set_field(f, a)
            np.testing.assert_array_equal(s.field(f), a)
            ldi, ldj = p.m + 5, p.n + 3
            wide = np.full(((p.l + 2) if p.dim == 3 else 1, ldj, ldi), -7.0)
            rc = lib().pf_download(s._h, FIELDS[f], wide.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), ldi, ldj)
            assert rc == 0
            np.testing.assert_array_equal(wide[:, :p.n + 2, :p.m + 2].reshape(shape), a)
            assert (wide[:, p.n + 2:, :] == -7.0).all() and (wide[:, :, p.m + 2:] == -7.0).all()
