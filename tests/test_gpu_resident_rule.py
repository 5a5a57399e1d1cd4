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


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_coefficient_bytes(precision, monkeypatch):
    """One set of 7 * 64 values for each wave, colour and height pair with a cell that is not unit:
    none for a porosity of 1, one cell of another needs a set for itself and for each neighbour's
    wave and pair, and a porosity that is nowhere 1 the whole grid's."""
    from pixelflow_amd.solver import PF_PREC_FP64, PF_PREC_MIXED, Solver
    monkeypatch.setenv("PF_RESIDENT", "2,1,2")       # 32x32x16 tiles: sixteen waves, eight pairs
    p, phi = _case("uniform", (64, 32, 32), 20, 1)
    one = 7 * 64 * (8 if precision == "fp64" else 4)
    kw = dict(precision=PF_PREC_MIXED if precision == "mixed" else PF_PREC_FP64)
    for value, sets in (("none", 0), ("one", 7), ("all", 4 * 16 * 8 * 2)):
        phi[:] = 0.5 if value == "all" else 1.0
        if value == "one":
            phi[11, 13, 40] = 0.5
        with Solver(p, phi, **kw) as s:
            assert s.sor_resident()
            got = s.resident_bytes()
            print(f"[gpu] coefficients {precision} {value} {got / one} sets", flush=True)
            if value == "one":
                assert 2 * one <= got <= sets * one        # cells of it share waves and pairs
                assert got > 7 * 7 * 8                      # more than its cells' own coefficients
            else:
                assert got == max(1, sets) * one            # the array is never empty
            assert got <= 7 * (8 if precision == "fp64" else 4) * p.cells


def test_the_parity_tests_solve_resident(monkeypatch):
    """The grids and tilings of test_gpu_resident.py are taken, for the whole of its steps (those
    of the rule's own choice that are too short for it excepted)."""
    from test_gpu_resident import RUNS, RUNS_2D, _case, _case_2d

    from pixelflow_amd.solver import PF_PREC_MIXED, Solver
    runs = [(r, dict(inner_iters=m * max(2, r[3] // 2), precision=m * PF_PREC_MIXED), lambda r=r: _case(r[0], r[1], r[3], 3), r[2])
            for r in RUNS for m in (0, 1)]
    runs += [(r, dict(inner_iters=m * r[2], precision=m * PF_PREC_MIXED), lambda r=r: _case_2d(r[0], r[2], 3, False), r[1])
             for r in RUNS_2D for m in (0, 1)]
    taken = 0
    for r, kw, make, forced in runs:
        if forced:
            monkeypatch.setenv("PF_RESIDENT", forced)
        else:
            monkeypatch.delenv("PF_RESIDENT", raising=False)
        p, phi = make()
        with Solver(p, phi, **kw) as s:
            before = s.sor_resident()
            s.step(3)
            assert s.sor_resident() == before
            assert before or not forced, (r, kw)
            taken += before
    assert taken >= len(runs) - 6, taken


def test_giving_up_between_cycles_and_coming_back(monkeypatch):
    """A mixed solve in three cycles a step: launches go well, then one gives up in the middle of
    the run, sixteen solves go by the sweeps, and the resident form takes over again; the bits
    are those of the sweeps throughout."""
    from pixelflow_amd.solver import PF_PREC_MIXED, Solver
    p, phi = _case("uniform", (64, 32, 31), 24, 12)
    kw = dict(precision=PF_PREC_MIXED, inner_iters=8)
    monkeypatch.setenv("PF_RESIDENT", "0")
    with Solver(p, phi, **kw) as s:
        ref = [np.concatenate([s.step(1)["sor_error"] for _ in range(12)])] + [s.field(f) for f in ("u", "v", "w", "p")]
    monkeypatch.setenv("PF_RESIDENT", "2,1,2")
    with Solver(p, phi, **kw) as s:
        errors = [s.step(1)["sor_error"] for _ in range(2)]
        assert s.sor_resident()
        monkeypatch.setenv("PF_RESIDENT_POLLS", "1")
        errors.append(s.step(1)["sor_error"])             # the first cycle gives up, two more pause
        assert not s.sor_resident()
        monkeypatch.delenv("PF_RESIDENT_POLLS")
        errors += [s.step(1)["sor_error"] for _ in range(4)]
        assert not s.sor_resident()                         # 14 of 16
        errors += [s.step(1)["sor_error"] for _ in range(5)]   # back within the first cycle pair
        assert s.sor_resident()
        out = [np.concatenate(errors)] + [s.field(f) for f in ("u", "v", "w", "p")]
    for a, b in zip(ref, out):
        np.testing.assert_array_equal(a, b)
