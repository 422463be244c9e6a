"""The solver settings of a cavity's steps: those of the first step whose solve
starts warm after the first two, as fdmgpu_ns_get documents, however the steps are
launched.  Bitwise against a run whose settings are never touched."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("calls", [(6,), (1, 1, 1, 1, 1, 1), (4, 2)])
def test_settings_kept(calls):
    import fdm_amd
    print("[case] cavity settings", calls, flush=True)
    a, b = (fdm_amd.NSCube(nx=31, ny=31, nz=31, Re=100.0, dt=0.01, solver="refine") for _ in range(2))
    a.step(4)
    b.step(4)
    b.set_solver_refine(1e-2, 2)
    for n in calls:
        a.step(n)
        b.step(n)
    for f in "uvwp":
        assert np.array_equal(a.get(f), b.get(f)), f
