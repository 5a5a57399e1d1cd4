"""Which solves are resident by the rule's own choice, and that those that are give the bits of
the oracle: tilings of the rule for both precisions at the edges of its ranges (the smallest
grids, odd extents, sixteen FP32 height pairs with a ragged last tile, rooms), and iteration
counts on either side of the least that it takes."""
import numpy as np
import pytest

from pixelflow_amd import cases

pytestmark = pytest.mark.gpu


def _case(kind, size, iters, steps):
    m, n, l = size
    if kind == "room":
        return cases.room_case(7, steps=steps, iter_max=iters, size=size)
    dx = 0.01
    p = cases.CaseParams(dim=3 if l > 1 else 2, m=m, n=n, l=l, width=dx * (m - 1), height=dx * (n - 1),
                         depth=dx * (l - 1) if l > 1 else 0.0, time=1e-4 * steps, istep_max=steps, iter_max=iters)
    rng = np.random.default_rng(m * n + l)
    phi = np.ones(p.interior_shape())
    some = rng.random(phi.shape) < 0.02
    phi[some] = rng.uniform(0.0, 1.0, int(some.sum()))
    return p, phi


FP64 = [
    ("uniform", (3, 3, 3), 6), ("uniform", (33, 27, 19), 7), ("uniform", (64, 30, 31), 6),
    ("room", (51, 88, 52), 6), ("room", (105, 113, 87), 8), ("uniform", (97, 65, 49), 6),
    ("uniform", (131, 97, 61), 8),
    ("uniform", (97, 51, 1), 6), ("uniform", (130, 40, 1), 12), ("uniform", (700, 300, 1), 12), ("uniform", (48, 24, 1), 2),
]


@pytest.mark.parametrize("kind,size,iters", FP64)
def test_rule_fp64(kind, size, iters, monkeypatch):
    import pyoracle
    from pixelflow_amd.solver import Solver
    print(f"[gpu] resident by rule {kind} {size} iters={iters}", flush=True)
    p, phi = _case(kind, size, iters, 2)
    o = pyoracle.OracleRun(p, phi)
    ref = o.step(2)
    with Solver(p, phi) as s:
        assert s.sor_resident()
        st = s.step(2)
        assert s.sor_resident()
        for f in ("u", "v", "w", "p") if p.dim == 3 else ("u", "v", "p"):
            np.testing.assert_array_equal(s.interior(f), o.interior(f), err_msg=f)
        np.testing.assert_array_equal(st["sor_error"], ref)


FP32 = [
    ("uniform", (3, 3, 3), "", 6), ("uniform", (33, 27, 19), "", 7), ("room", (105, 113, 87), "", 12),
    ("uniform", (131, 97, 61), "", 12),
    ("uniform", (64, 60, 93), "2,2,3", 5),       # sixteen height pairs, the last tile ragged
    ("uniform", (63, 61, 93), "2,2,3", 5),       # the same with odd extents
    ("room", (64, 60, 91), "2,2,3", 5),          # and with a room's walls
    ("uniform", (30, 29, 31), "1,1,1", 4),       # one tile of sixteen, its own neighbour
]


@pytest.mark.parametrize("kind,size,tiles,iters", FP32)
def test_rule_mixed(kind, size, tiles, iters, monkeypatch):
    from pixelflow_amd.solver import PF_PREC_MIXED, Solver
    p, phi = _case(kind, size, 2 * iters + 1, 2)   # two cycles a step and one of a single iteration
    out = []
    for mode in (tiles, "0"):
        if mode:
            monkeypatch.setenv("PF_RESIDENT", mode)
        print(f"[gpu] resident by rule, mixed {kind} {size} tiles={mode or 'rule'}", flush=True)
        with Solver(p, phi, precision=PF_PREC_MIXED, inner_iters=iters) as s:
            assert s.sor_resident() == (mode != "0")
            st = s.step(2)
            assert s.sor_resident() == (mode != "0")
            out.append([s.interior(f) for f in ("u", "v", "w", "p")] + [st["sor_error"]])
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("size,mixed,least", [((48, 40, 40), False, 6), ((48, 40, 40), True, 6), ((96, 96, 64), False, 8),
                                              ((96, 96, 64), True, 12), ((130, 40, 1), False, 12), ((131, 41, 1), False, 6)])
def test_short_solves_are_left_to_the_sweeps(size, mixed, least):
    from pixelflow_amd.solver import PF_PREC_FP64, PF_PREC_MIXED, Solver
    for iters in (least - 1, least):
        p, phi = _case("uniform", size, iters, 1)
        with Solver(p, phi, precision=PF_PREC_MIXED if mixed else PF_PREC_FP64) as s:
            assert s.sor_resident() == (iters >= least)
