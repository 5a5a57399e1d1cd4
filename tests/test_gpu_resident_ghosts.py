"""Resident 3D solves from a pressure whose ghost cells are no mirrors of the grid's own (an
uploaded field keeps the ghosts it came with): the first half-sweep takes them as they are, all
later ones the cells they mirror.  Across an odd periodic extent a ghost has its reader's
colour.  Against the per-half-sweep kernels, bit for bit."""
import numpy as np
import pytest

from pixelflow_amd import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("size,tiles", [
    ((33, 26, 18), "2,2,3"),      # even extents
    ((33, 27, 18), "2,2,3"),      # odd in y
    ((33, 26, 19), "2,2,3"),      # odd in z
    ((33, 27, 19), "2,2,3"),      # odd in both
    ((30, 27, 7), "1,1,1"),       # the same within one tile, its own neighbour
    ((45, 29, 9), "2,1,9"),       # one-cell-thick tiles
])
def test_uploaded_ghosts(size, tiles, precision, monkeypatch):
    from pixelflow_amd.solver import PF_PREC_FP64, PF_PREC_MIXED, Solver
    m, n, l = size
    dx = 0.01
    p = cases.CaseParams(dim=3, m=m, n=n, l=l, width=dx * (m - 1), height=dx * (n - 1), depth=dx * (l - 1),
                         time=2e-4, istep_max=2, iter_max=6)
    rng = np.random.default_rng(m * n + l)
    phi = np.ones((l, n, m))
    some = rng.random(phi.shape) < 0.05
    phi[some] = rng.uniform(0.0, 1.0, int(some.sum()))
    kw = dict(precision=PF_PREC_MIXED, inner_iters=3) if precision == "mixed" else dict(precision=PF_PREC_FP64)
    pressure = rng.standard_normal(p.full_shape())
    out = []
    for mode in ("0", tiles):
        monkeypatch.setenv("PF_RESIDENT", mode)
        print(f"[gpu] uploaded ghosts {size} {precision} tiles={mode}", flush=True)
        with Solver(p, phi, **kw) as s:
            assert s.sor_resident() == (mode != "0")
            s.set_field("p", pressure)
            st = s.step(2)
            assert s.sor_resident() == (mode != "0")
            out.append([s.field(f) for f in ("u", "v", "w", "p")] + [st["sor_error"]])
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
