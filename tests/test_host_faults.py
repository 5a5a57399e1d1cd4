"""What the host code does when a HIP call fails or a resident launch gives up, on the CPU:
the library over a stand-in for the HIP runtime (tests/native/hip_stand_in.cpp) in a process
of its own.  No kernel computes anything there; the tests look at error codes, at which
kernels are launched, and at what is held afterwards."""
import os
import subprocess
import sys
import textwrap

import pytest

from pixelflow_amd import build, solver

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

pytestmark = pytest.mark.skipif(not os.path.exists(solver.LIB_PATH) or not os.path.exists(build.HIP_STAND_IN),
                                reason="HIP library or its stand-in not built (python -m pixelflow_amd.build)")

HEAD = """
import ctypes, os, sys, threading
import numpy as np
from pixelflow_amd import build, cases, solver as S
F = ctypes.CDLL(build.HIP_STAND_IN, mode=ctypes.RTLD_GLOBAL)   # before the library: its HIP calls go here
F.fake_allocated.restype = ctypes.c_size_t
F.fake_read.argtypes = [ctypes.c_void_p, ctypes.c_size_t]
def launches(part): return F.fake_launches(part.encode())
def fail(fn, skip=0, times=1, err=719): F.fake_fail(fn.encode(), skip, times, err)   # 719: hipErrorLaunchFailure
def calls(fn): return F.fake_calls(fn.encode())
def read(values, dtype="f8"):
    a = np.asarray(values, dtype=dtype)
    F.fake_read(a.ctypes.data, a.nbytes)
def case(size=(64, 32, 32), iters=40):
    m, n, l = size
    p = cases.CaseParams(dim=3 if l > 1 else 2, m=m, n=n, l=l, width=0.01 * (m - 1), height=0.01 * (n - 1),
                         depth=0.01 * (l - 1) if l > 1 else 0.0, time=1.0, istep_max=10**6, iter_max=iters)
    return p, np.ones(p.interior_shape())
def raises(f):
    try: f()
    except S.PixelFlowError as e: return str(e)
    return None
"""


def run(body, **env):
    r = subprocess.run([sys.executable, "-c", HEAD + textwrap.dedent(body) + "\nprint('ok')"], cwd=ROOT,
                       env=dict(os.environ, **env), capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout + r.stderr


@pytest.mark.parametrize("where", ["count copy", "resident wait"])
@pytest.mark.parametrize("kind", ["3d", "2d", "mixed", "tolerance"])
def test_a_failed_wait_for_a_resident_solve_fails_the_step(where, kind):
    """What the launch left is not known then: it may have written its result."""
    run(f"""
        kind, where = {kind!r}, {where!r}
        p, phi = case((64, 32, 1) if kind == "2d" else (64, 32, 32))
        if kind == "2d": os.environ["PF_RESIDENT"] = "1,2"
        kw = dict(precision=S.PF_PREC_MIXED, inner_iters=20) if kind == "mixed" else {{}}
        if kind == "tolerance":
            kw = dict(residual_tol=1e-9)
        with S.Solver(p, phi, **kw) as s:
            assert s.sor_resident()
            if kind == "tolerance": read([1.0])
            s.step(1)
            n = launches("k_sor_resident")
            assert n >= 1
            if kind == "tolerance": read([1.0])
            fail(where)
            msg = raises(lambda: s.step(1))
            assert msg and "PF_EHIP" in msg, msg
            assert launches("k_sor_resident") == n + 1
            assert not launches("k_sor_phi") and not launches("k_sor32") and not launches("k_sor_tb2")
    """)


@pytest.mark.parametrize("kind", ["3d", "2d", "mixed"])
def test_a_refused_launch_leaves_the_solve_to_the_sweeps(kind):
    run(f"""
        kind = {kind!r}
        p, phi = case((64, 32, 1) if kind == "2d" else (64, 32, 32))
        if kind == "2d": os.environ["PF_RESIDENT"] = "1,2"
        kw = dict(precision=S.PF_PREC_MIXED, inner_iters=20) if kind == "mixed" else {{}}
        with S.Solver(p, phi, **kw) as s:
            fail("resident launch")
            s.step(1)
            assert not launches("k_sor_resident")
            assert launches("k_sor_phi") + launches("k_sor32") + launches("k_sor_tb2")
    """)


@pytest.mark.parametrize("kind", ["3d", "2d", "mixed"])
def test_a_launch_that_gives_up_is_tried_again_after_a_pause(kind):
    """16 solves by the sweeps (in 2D FP64 the blocked one), 32 after the next time,
    and from then on resident again."""
    run(f"""
        kind = {kind!r}
        p, phi = case((64, 32, 1) if kind == "2d" else (64, 32, 32))
        if kind == "2d": os.environ["PF_RESIDENT"] = "1,2"
        kw = dict(precision=S.PF_PREC_MIXED, inner_iters=40) if kind == "mixed" else {{}}
        sweep = {{"3d": "k_sor_phi", "2d": "k_sor_tb2", "mixed": "k_sor32"}}[kind]
        with S.Solver(p, phi, **kw) as s:
            F.fake_give_up(2)
            tries, solves = [], []
            for step in range(80):
                a, b = launches("k_sor_resident"), launches(sweep)
                s.step(1)
                if launches("k_sor_resident") > a: tries.append(step)
                assert (launches(sweep) > b) == (step < 50), step   # 0..16 and 17..49
                assert s.sor_resident() == (step in (16, 49) or step > 49), step
            assert tries == [0, 17] + list(range(50, 80)), tries
            F.fake_give_up(1)
            for step in range(65):   # after 30 good solves of the 32 the pause doubles
                s.step(1)
            assert launches("k_sor_resident") == len(tries) + 1
    """)


@pytest.mark.parametrize("tiles,together", [
    ("2,1,2", 2),     # a few CUs each: both at once
    ("8,4,8", 1),     # 256 blocks of a whole CU each: one after the other
])
def test_resident_launches_of_two_threads_share_the_chip(tiles, together):
    run(f"""
        os.environ["PF_RESIDENT"] = {tiles!r}
        size = (64, 32, 32) if {together} == 2 else (256, 128, 128)
        p, phi = case(size)
        solvers = [S.Solver(p, phi) for _ in range(2)]
        assert all(s.sor_resident() for s in solvers)
        F.fake_hold(50)
        threads = [threading.Thread(target=s.step, args=(3,)) for s in solvers]
        for t in threads: t.start()
        for t in threads: t.join()
        assert F.fake_most_resident() == {together}, F.fake_most_resident()
        assert launches("k_sor_resident") == 6 and not launches("k_sor_phi")
    """)


def test_resident_launches_take_turns_in_the_order_of_asking():
    """A launch that needs the whole chip gets it although smaller ones keep coming."""
    run("""
        import time
        os.environ["PF_RESIDENT"] = "2,1,2"
        small = [S.Solver(*case((64, 32, 32))) for _ in range(3)]
        os.environ["PF_RESIDENT"] = "8,4,8"
        large = S.Solver(*case((256, 128, 128)))
        F.fake_hold(20)
        stop = threading.Event()
        def keep(s):
            while not stop.is_set(): s.step(1)
        threads = [threading.Thread(target=keep, args=(s,)) for s in small]
        for t in threads: t.start()
        time.sleep(0.1)
        t0 = time.perf_counter()
        large.step(2)
        took = time.perf_counter() - t0
        stop.set()
        for t in threads: t.join()
        assert took < 5.0, took
    """)


@pytest.mark.parametrize("kind", ["3d", "2d", "mixed"])
def test_no_room_for_the_resident_form_leaves_the_sweeps(kind):
    """Each allocation of pf_create fails once: those of the resident form leave a context that
    solves by the sweeps, any other fails the call; nothing is left behind."""
    run(f"""
        kind = {kind!r}
        p, phi = case((130, 40, 1) if kind == "2d" else (64, 32, 32))
        kw = dict(precision=S.PF_PREC_MIXED, inner_iters=20) if kind == "mixed" else {{}}
        def mallocs(mode):
            os.environ["PF_RESIDENT"] = mode
            F.fake_reset()
            S.Solver(p, phi, **kw).close()
            os.environ.pop("PF_RESIDENT")
            return calls("hipMalloc")
        own = mallocs("") - mallocs("0")
        own -= 1 if kind != "2d" else 0      # the coefficients, of pf_set_porosity
        assert own == (2 if kind == "2d" else 4), own
        n, sweeps = mallocs(""), 0
        for at in range(n):
            F.fake_reset()
            fail("hipMalloc", skip=at, err=2)   # hipErrorOutOfMemory
            try:
                s = S.Solver(p, phi, **kw)
            except S.PixelFlowError as e:
                assert "PF_ENOMEM" in str(e) or "PF_EHIP" in str(e), e
            else:
                sweeps += not s.sor_resident()
                s.step(2)
                assert bool(launches("k_sor_resident")) == s.sor_resident()
                s.close()
            assert F.fake_allocated() == 0, at
        assert sweeps == own + (kind != "2d"), sweeps
        F.fake_reset()
        fail("hipHostMalloc", err=2)
        with S.Solver(p, phi, **kw) as s:
            assert not s.sor_resident()
            s.step(2)
        assert F.fake_allocated() == 0
    """)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_a_porosity_that_was_not_set_up_is_not_solved_resident(precision):
    """pf_set_porosity fails before the masks and coefficients are those of one porosity: a later
    step does not launch on them; with a porosity that was set up it does again."""
    run(f"""
        kw = dict(precision=S.PF_PREC_MIXED, inner_iters=20) if {precision!r} == "mixed" else {{}}
        p, phi = case()
        raw = np.random.default_rng(1).random(phi.size)
        failed = 0
        for fn in ("hipMemcpyAsync", "hipStreamSynchronize"):
            for at in range(12):
                F.fake_reset()
                with S.Solver(p, phi, **kw) as s:
                    s.step(1)
                    assert s.sor_resident() and launches("k_sor_resident")
                    F.fake_reset()
                    fail(fn, skip=at)
                    rc = S.lib().pf_set_porosity(s._h, S._dp(raw), float(p.threshold))
                    if rc == 0 or launches("k_resident_setup") > 1: continue   # none failed, or a later one
                    failed += 1
                    F.fake_reset()
                    assert not s.sor_resident(), (fn, at)
                    s.step(1)
                    assert not launches("k_sor_resident"), (fn, at)
                    s._check(S.lib().pf_set_porosity(s._h, S._dp(raw), float(p.threshold)), "pf_set_porosity")
                    s.step(1)
                    assert s.sor_resident() and launches("k_sor_resident")
        assert failed >= 6, failed
    """)


@pytest.mark.parametrize("call", ["hipGraphLaunch", "hipGraphInstantiate", "hipStreamBeginCapture", "hipStreamEndCapture"])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_a_graph_that_fails_leaves_the_iteration_to_launches(call, precision):
    """A batch's multigrid solves launch an iteration as one graph; where that fails the kernels
    are launched one by one, the step succeeds and the graph is not tried again."""
    run(f"""
        kw = dict(residual_tol=1e-9, solver=S.PF_SOLVER_MG, max_cycles=30)
        if {precision!r} == "mixed": kw["precision"] = S.PF_PREC_MIXED
        p, phi = case((16, 16, 16))
        arena = 2 * S.batch_case_bytes(p, **kw) + (64 << 20)
        b = S.Batch(p, max_cases=2, arena_bytes=arena, **kw)
        for _ in range(2): b.add(p, phi)
        def step():   # residual 1, an inner solve that ends after one iteration, residual 0; per case
            for v in (1.0, 1.0, 0.0, 0.0): read([v])
            for _ in range(2): read([0, 0, 0, 0, 1.0, 1.0, 0, 0])
            for _ in range(2): read([0, 0, 0, 0, 1.0, 0.0, 0, 0])
            b.step(1)
        step()
        assert launches("graph") == 2, launches("graph")
        b.close()
        F.fake_reset()
        b = S.Batch(p, max_cases=2, arena_bytes=arena, **kw)
        for _ in range(2): b.add(p, phi)
        fail({call!r}, times=2)
        step()
        assert not launches("graph") and launches("k_bicg_xr") == 2, (launches("graph"), launches("k_bicg_xr"))
        step()
        assert not launches("graph") and launches("k_bicg_xr") == 4
        b.close()
    """)


@pytest.mark.parametrize("call", ["hipHostMalloc", "hipEventCreateWithFlags"])
@pytest.mark.parametrize("dim", [2, 3])
def test_fields_come_without_pinned_memory(call, dim):
    run(f"""
        os.environ["PF_RESIDENT"] = "0"
        p, phi = case((33, 21, 1) if {dim} == 2 else (33, 21, 13))
        rng = np.random.default_rng(2)
        s = S.Solver(p, phi)
        b = S.Batch(p, max_cases=1, arena_bytes=S.batch_case_bytes(p) + (64 << 20))
        slot = b.add(p, phi)
        fail({call!r}, times=-1)
        for f in ("u", "v", "p"):
            a = rng.standard_normal(p.full_shape())
            s.set_field(f, a)
            np.testing.assert_array_equal(s.field(f), a)
            assert b.field(slot, f).shape == p.full_shape()
            assert F.hipGetLastError() == 0
        assert not launches("k_pack")
        ldi, ldj = p.m + 5, p.n + 3
        wide = np.full((p.l + 2 if {dim} == 3 else 1, ldj, ldi), -7.0)
        assert S.lib().pf_download(s._h, S.FIELDS["p"], S._dp(wide), ldi, ldj) == 0
        np.testing.assert_array_equal(wide[:, :p.n + 2, :p.m + 2].reshape(p.full_shape()), a)
        assert (wide[:, p.n + 2:, :] == -7.0).all() and (wide[:, :, p.m + 2:] == -7.0).all()
    """)


def test_fields_of_one_context_in_several_threads():
    run("""
        os.environ["PF_RESIDENT"] = "0"
        p, phi = case((33, 21, 13))
        s = S.Solver(p, phi)
        values = {"u": 1.0, "v": 2.0, "w": 3.0, "p": 4.0}
        for f, v in values.items(): s.set_field(f, np.full(p.full_shape(), v))
        F.fake_hold(1)
        wrong = []
        def keep(f):
            for _ in range(20):
                if not (s.field(f) == values[f]).all(): wrong.append(f)
        threads = [threading.Thread(target=keep, args=(f,)) for f in values]
        for t in threads: t.start()
        for t in threads: t.join()
        assert not wrong, wrong
    """)


@pytest.mark.parametrize("kind", ["3d", "2d"])
def test_message_numbers_start_over_on_an_empty_inbox(kind):
    """Numbers are 32 bits; before they run out the inbox is cleared and they begin again."""
    run(f"""
        if {kind!r} == "2d": os.environ["PF_RESIDENT"] = "1,2"
        p, phi = case((64, 32, 1) if {kind!r} == "2d" else (64, 32, 32), iters=(1 << 28) - 1)
        used, cleared = 1, 0
        with S.Solver(p, phi) as s:
            for step in range(40):
                a = launches("k_clear_u64")
                s.step(1)
                need = p.iter_max if {kind!r} == "2d" else 2 * p.iter_max
                over = used + need > 0xffffffff
                used = need + (1 if over else used)
                cleared += over
                assert launches("k_clear_u64") - a == 1 + over, step     # the step's own and the inbox
            assert cleared >= 2 and launches("k_sor_resident") == 40
    """)


def test_a_cycle_that_gives_up_is_swept_alone():
    """The second of three cycles of a step: one cycle's sweeps and one update each, then a pause."""
    run("""
        p, phi = case(iters=60)
        with S.Solver(p, phi, precision=S.PF_PREC_MIXED, inner_iters=20) as s:
            F.fake_give_up_after(1, 1)
            n = launches("k_update")
            s.step(1)
            assert launches("k_sor_resident") == 2            # the first, and the one that gave up
            assert launches("k_sor32") == 2 * 2 * 20           # the second and the third
            assert launches("k_update") - n == 3
            for _ in range(5): s.step(1)                        # fifteen more of the pause
            assert launches("k_sor_resident") == 2
            s.step(1)
            assert launches("k_sor_resident") == 5
    """)
