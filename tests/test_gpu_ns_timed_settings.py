"""A timed step of the cavity takes the solver settings of the untimed steps
around it (those of the first step whose solve starts warm after the first two), as
fdmgpu_ns_step_timed documents, and so do steps replayed from a graph.  Bitwise
against a run whose settings are never touched."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def pair(solver, n=31):
    import fdm_amd
    return [fdm_amd.NSCube(nx=n, ny=n, nz=n, Re=100.0, dt=0.01, solver=solver) for _ in range(2)]


def run(ns, calls):
    for n in calls:
        if n == "timed":
            ns.step_timed()
        else:
            ns.step(n)


def same(a, b):
    for f in "uvwp":
        assert np.array_equal(a.get(f), b.get(f)), f


def set_variant(ns, v):
    import fdm_amd
    plan = ctypes.c_void_p()
    assert fdm_amd.lib().fdmgpu_ns_solver(ns._h, ctypes.byref(plan)) == 0
    assert fdm_amd.lib().fdmgpu_plan_set_variant(plan, ctypes.byref(fdm_amd.Variant(*v))) == 0


@pytest.mark.parametrize("calls", [("timed",), ("timed", 1, "timed", 3), (2, "timed", 1)])
@pytest.mark.parametrize("first", [(4,), (2, "timed"), ("timed", 1, 1)])
def test_refine_settings(first, calls):
    print("[case] cavity timed settings", first, calls, flush=True)
    a, b = pair("refine")
    for ns in (a, b):
        run(ns, first)
    b.set_solver_refine(1e-2, 2)
    for ns in (a, b):
        run(ns, calls)
    same(a, b)


# single steps of a small FP64 grid are replayed, longer calls and timed steps are not
@pytest.mark.parametrize("first,calls", [((4,), (1, "timed", 2, 1)), ((1, 1, 1, 1), (2, 1, "timed")),
                                         ((2, "timed"), (1, 1, 3))])
def test_f64_variant(first, calls):
    print("[case] cavity variant", first, calls, flush=True)
    a, b = pair("f64")
    for ns in (a, b):
        run(ns, first)
    set_variant(b, (0, 16, 16, 1, 0))
    for ns in (a, b):
        run(ns, calls)
    same(a, b)


def test_settings_matter():
    """(the runs above would differ if a step took the changed settings)"""
    a, b = pair("refine")
    b.set_solver_refine(1e-2, 2)
    run(a, (4,))
    run(b, (4,))
    assert not np.array_equal(a.get("p"), b.get("p"))
    a, b = pair("f64")
    set_variant(b, (0, 16, 16, 1, 0))
    run(a, (4,))
    run(b, (4,))
    assert not np.array_equal(a.get("p"), b.get("p"))
