"""The coarse end of the multigrid cycle as launches (restriction by one lane per fine cell, the
coarsest solve over several blocks) against the same cycle inside one block, which sums in the
same order: bit for bit, over even and odd extents, aggregates cut by the grid's edge, coarsest
levels that are no multiple of a block's rows, two and three dimensions, and the rooms."""
import numpy as np
import pytest

from pixelflow_amd import cases

pytestmark = pytest.mark.gpu


def _case(kind, size):
    m, n, l = size
    if kind == "room":
        return cases.room_case(3, steps=2, size=size)
    dx = 0.01
    p = cases.CaseParams(dim=3 if l > 1 else 2, m=m, n=n, l=l, width=dx * (m - 1), height=dx * (n - 1),
                         depth=dx * (l - 1) if l > 1 else 0.0, time=2e-4, istep_max=2, iter_max=20)
    phi = np.ones(p.interior_shape())
    some = np.random.default_rng(m + n + l).random(phi.shape) < 0.03
    phi[some] = 0.3
    return p, phi


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("kind,size", [("uniform", (64, 48, 40)), ("uniform", (65, 33, 17)), ("uniform", (30, 18, 11)),
                                       ("uniform", (97, 51, 1)), ("uniform", (128, 64, 1)), ("room", (48, 40, 33))])
def test_coarse_launches_match_the_one_block_cycle(kind, size, precision, monkeypatch):
    from pixelflow_amd.solver import PF_PREC_FP64, PF_PREC_MIXED, PF_SOLVER_MG, Solver
    p, phi = _case(kind, size)
    out = []
    for tail in (None, "8192"):
        if tail:
            monkeypatch.setenv("PF_MG_TAIL", tail)
        print(f"[gpu] coarse cycle {kind} {size} {precision} tail={tail}", flush=True)
        with Solver(p, phi, precision=PF_PREC_MIXED if precision == "mixed" else PF_PREC_FP64, residual_tol=1e-9,
                    solver=PF_SOLVER_MG, max_cycles=30) as s:
            st = s.step(2)
            fields = ("u", "v", "w", "p") if p.dim == 3 else ("u", "v", "p")
            out.append([s.interior(f) for f in fields] + [st["residual"]])
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
