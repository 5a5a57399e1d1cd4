"""Solves run as one launch with the grid resident on chip (pf_resident.hip).

FP64 against the oracle bit for bit, the FP32 correction sweeps against the per-half-sweep
kernels bit for bit (the same operations on the same operands), over tilings with one and
many tiles per axis, ragged last tiles, one to sixteen height pairs per thread, even and odd
periodic extents (an odd one wraps a colour onto itself) and the rooms' walls.
"""
import numpy as np
import pytest

from pixelflow_amd import cases

pytestmark = pytest.mark.gpu


def _case(bc, size, iters, steps):
    m, n, l = size
    if bc == "air":
        return cases.room_case(5, steps=steps, iter_max=iters, size=size)
    dx = 0.01
    p = cases.CaseParams(dim=3, m=m, n=n, l=l, width=dx * (m - 1), height=dx * (n - 1), depth=dx * (l - 1),
                         time=1e-4 * steps, istep_max=steps, iter_max=iters)
    rng = np.random.default_rng(m * n + l)
    phi = np.ones((l, n, m))
    some = rng.random(phi.shape) < 0.01          # isolated cells, so unit and other waves both occur
    phi[some] = rng.uniform(0.0, 1.0, int(some.sum()))
    phi[l // 3:l // 2, n // 3:n // 2, m // 3:m // 2] = rng.uniform(0.0, 1.0)
    return p, phi


RUNS = [
    ("uniform", (64, 32, 32), "2,1,2", 7),       # 32x32 tiles, eight height pairs
    ("uniform", (64, 32, 32), "4,2,8", 6),
    ("uniform", (33, 27, 19), "2,2,3", 5),       # odd periodic extents, ragged tiles
    ("uniform", (45, 28, 9), "2,1,9", 4),        # one-cell-thick tiles, a tile its own neighbour in y
    ("uniform", (30, 32, 7), "1,1,1", 3),        # a single tile, its own neighbour in y and z
    ("uniform", (41, 21, 16), "3,4,2", 2),       # the fewest iterations of a resident solve
    ("uniform", (97, 65, 49), "", 9),            # the rule's own tiling
    ("air", (64, 48, 40), "2,2,3", 6),
    ("air", (48, 40, 33), "", 5),
]


@pytest.mark.parametrize("bc,size,tiles,iters", RUNS)
def test_resident_solve_matches_oracle(bc, size, tiles, iters, monkeypatch):
    import pyoracle
    from pixelflow_amd.solver import Solver
    if tiles:
        monkeypatch.setenv("PF_RESIDENT", tiles)
    print(f"[gpu] resident {bc} {size} tiles={tiles or 'rule'} iters={iters}", flush=True)
    p, phi = _case(bc, size, iters, 3)
    o = pyoracle.OracleRun(p, phi)
    ref = o.step(3)
    with Solver(p, phi) as s:
        st = s.step(3)
        for f in ("u", "v", "w", "p"):
            np.testing.assert_array_equal(s.interior(f), o.interior(f), err_msg=f)
        np.testing.assert_array_equal(st["sor_error"], ref)


@pytest.mark.parametrize("bc,size,tiles,iters", RUNS + [("uniform", (64, 64, 64), "2,2,2", 6)])
def test_resident_fp32_solve_matches_sweeps(bc, size, tiles, iters, monkeypatch):
    from pixelflow_amd.solver import PF_PREC_MIXED, Solver
    p, phi = _case(bc, size, iters, 3)
    out = {}
    for mode in ("0", tiles):
        if mode:
            monkeypatch.setenv("PF_RESIDENT", mode)
        else:
            monkeypatch.delenv("PF_RESIDENT")
        print(f"[gpu] resident FP32 {bc} {size} tiles={mode or 'rule'} iters={iters}", flush=True)
        with Solver(p, phi, precision=PF_PREC_MIXED, inner_iters=max(2, iters // 2)) as s:
            st = s.step(3)
            out[mode == "0"] = [s.interior(f) for f in ("u", "v", "w", "p")] + [st["sor_error"]]
    for a, b in zip(out[True], out[False]):
        np.testing.assert_array_equal(a, b)


RUNS_2D = [
    ((48, 24), "", 9),           # one block holds the grid
    ((48, 23), "", 9),           # the same with an odd extent in y
    ((37, 12), "1,2", 7),        # two rows a block, an exchange per iteration
    ((37, 13), "1,2", 7),        # odd extent, the last block one row short
    ((130, 40), "2,3", 9),       # two iterations between exchanges, ragged last block and round
    ((131, 41), "3,1", 10),
    ((97, 51), "", 40),
    ((511, 255), "", 12),
    ((700, 300), "", 5),
    ((64, 32), "4,1", 8),        # as few rounds as a resident solve takes
]


@pytest.mark.parametrize("size,plan,iters", RUNS_2D)
@pytest.mark.parametrize("step", [False, True])
def test_resident_2d_solve_matches_oracle(size, plan, iters, step, monkeypatch):
    import pyoracle
    from pixelflow_amd.solver import Solver
    if plan:
        monkeypatch.setenv("PF_RESIDENT", plan)
    print(f"[gpu] resident 2D {size} plan={plan or 'rule'} iters={iters} step={step}", flush=True)
    p, phi = _case_2d(size, iters, 3, step)
    o = pyoracle.OracleRun(p, phi)
    ref = o.step(3)
    with Solver(p, phi) as s:
        st = s.step(3)
        for f in ("u", "v", "p"):
            np.testing.assert_array_equal(s.interior(f), o.interior(f), err_msg=f)
        np.testing.assert_array_equal(st["sor_error"], ref)


@pytest.mark.parametrize("size,plan,iters", RUNS_2D)
def test_resident_2d_fp32_solve_matches_sweeps(size, plan, iters, monkeypatch):
    """Also from ghost rows that are no mirrors of the grid's own (an uploaded pressure)."""
    from pixelflow_amd.solver import PF_PREC_FP64, PF_PREC_MIXED, Solver
    p, phi = _case_2d(size, iters, 3, False)
    for prec in (PF_PREC_MIXED, PF_PREC_FP64):
        out = {}
        for mode in ("0", plan):
            if mode:
                monkeypatch.setenv("PF_RESIDENT", mode)
            else:
                monkeypatch.delenv("PF_RESIDENT")
            monkeypatch.setenv("PF_SOR_TB2", "0,0") if mode == "0" else monkeypatch.delenv("PF_SOR_TB2")
            print(f"[gpu] resident 2D sweeps {size} plan={mode or 'rule'} prec={prec}", flush=True)
            with Solver(p, phi, precision=prec, inner_iters=iters if prec == PF_PREC_MIXED else 0) as s:
                s.set_field("p", np.random.default_rng(3).standard_normal(p.full_shape()))
                st = s.step(3)
                out[mode == "0"] = [s.interior(f) for f in ("u", "v", "p")] + [st["sor_error"]]
        for a, b in zip(out[True], out[False]):
            np.testing.assert_array_equal(a, b)


def _case_2d(size, iters, steps, step):
    m, n = size
    dx = 0.01
    p = cases.CaseParams(dim=2, m=m, n=n, width=dx * (m - 1), height=dx * (n - 1), time=1e-4 * steps, istep_max=steps,
                         iter_max=iters, inlet_porosity=step)
    rng = np.random.default_rng(m * n)
    phi = np.ones((n, m))
    some = rng.random(phi.shape) < 0.1
    phi[some] = rng.uniform(0.0, 1.0, int(some.sum()))
    return p, phi


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("dim", [2, 3])
def test_a_launch_that_gives_up_leaves_the_solve_to_the_sweeps(dim, precision, monkeypatch):
    """A wait of one poll: blocks give up, the launch changes nothing, and the context solves on
    with the per-half-sweep kernels."""
    from pixelflow_amd.solver import PF_PREC_FP64, PF_PREC_MIXED, Solver
    p, phi = _case_2d((130, 40), 8, 3, False) if dim == 2 else _case("uniform", (64, 32, 32), 8, 3)
    kw = dict(precision=PF_PREC_MIXED, inner_iters=8) if precision == "mixed" else dict(precision=PF_PREC_FP64)
    fields = ("u", "v", "p") if dim == 2 else ("u", "v", "w", "p")
    out = []
    for polls in (None, "1"):
        if polls:
            monkeypatch.setenv("PF_RESIDENT_POLLS", polls)
        monkeypatch.setenv("PF_RESIDENT", "1,2" if dim == 2 else "2,1,2")
        with Solver(p, phi, **kw) as s:
            assert s.sor_resident()
            st = s.step(3)
            assert s.sor_resident() == (polls is None)
            out.append([s.interior(f) for f in fields] + [st["sor_error"]])
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


def test_resident_contexts_in_two_threads():
    """Two contexts, each of whose solves takes every CU, stepped from two threads at once."""
    import threading

    from pixelflow_amd.solver import Solver
    p, phi = cases.sphere_case(m=256, n=128, l=128, steps=4, iter_max=10)
    with Solver(p, phi) as s:
        assert s.sor_resident()
        s.step(4)
        ref = s.interior("p")
    out, errors = [None, None], []

    def run(q):
        try:
            with Solver(p, phi) as s:
                s.step(4)
                out[q] = s.interior("p")
        except Exception as e:   # reported by the main thread
            errors.append(e)

    print("[gpu] resident contexts in two threads", flush=True)
    threads = [threading.Thread(target=run, args=(q,)) for q in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    for x in out:
        np.testing.assert_array_equal(x, ref)
