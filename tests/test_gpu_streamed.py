"""The per-half-sweep kernels on the grids whose solves are resident by default: the path of
larger grids, of short solves and of a context whose launch gave up.  FP64 against the reference's
fixtures and the oracle bit for bit, several steps, with the launch settings of these sizes."""
import numpy as np
import pytest

from conftest import load_golden
from test_gpu_parity import CASES, FULL, _fields, _solver, _sparse_porosity

from pixelflow_amd import cases

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _no_resident_solves(monkeypatch):
    monkeypatch.setenv("PF_RESIDENT", "0")


@pytest.mark.parametrize("name", FULL)
def test_streamed_matches_reference_fixture(name):
    p, g = load_golden(name)
    print(f"[gpu] streamed fixture {name}", flush=True)
    with _solver(p, g["phi_raw"]) as s:
        assert not s.sor_resident()
        st = s.step(p.istep_max)
        for f in _fields(p):
            np.testing.assert_array_equal(s.interior(f), g[f], err_msg=f"{name}:{f}")
        np.testing.assert_array_equal(st["sor_error"], g["errs"], err_msg=f"{name}:errs")


@pytest.mark.parametrize("name", sorted(CASES) + ["sparse"])
def test_streamed_matches_oracle(name):
    import pyoracle
    if name == "sparse":
        p = cases.CaseParams(dim=3, m=134, n=34, l=22, width=1.34, height=0.34, depth=0.22, time=3e-4, istep_max=3,
                             iter_max=20)
        phi = _sparse_porosity(p, 11)
    else:
        p, phi = CASES[name]()
    print(f"[gpu] streamed oracle case {name}", flush=True)
    o = pyoracle.OracleRun(p, phi)
    ref = o.step(p.istep_max)
    with _solver(p, phi) as s:
        assert not s.sor_resident()
        if name == "sparse":
            assert 0 < s.sor_unit_cells() < p.cells     # the flags that the sweeps read
        st = s.step(p.istep_max)
        np.testing.assert_array_equal(st["sor_error"], ref)
        for f in _fields(p):
            np.testing.assert_array_equal(s.interior(f), o.interior(f), err_msg=f"{name}:{f}")
