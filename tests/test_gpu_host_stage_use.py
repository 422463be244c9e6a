"""Which host arrays go through the host stage (host_stage.hip): pageable ones do,
seen by its threads, which are made for a plan's second solve, take part and end with
the plan; pinned ones, which the runtime copies at the link's rate, do not."""
import ctypes
import os
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def plan(n, precision="f64"):
    import fdm_amd
    h = [2 * np.pi / m for m in n]
    return fdm_amd.LaplCube(*h, *[(m + 1) * v for m, v in zip(n, h)], *n, precision=precision)


def threads():
    return set(os.listdir("/proc/self/task"))


def busy(tids):
    """Nanoseconds on a CPU, summed over the threads."""
    return sum(int(open("/proc/self/task/%s/schedstat" % t).read().split()[0]) for t in tids)


class Pinned:
    def __init__(self, shape, dtype):
        from fdm_amd import hip
        self.rt, self.p = hip.rt(), ctypes.c_void_p()
        nbytes = int(np.prod(shape)) * np.dtype(dtype).itemsize
        self.rt.hipHostMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t, ctypes.c_uint]
        assert self.rt.hipHostMalloc(ctypes.byref(self.p), nbytes, 0) == 0
        self.a = np.frombuffer((ctypes.c_char * nbytes).from_address(self.p.value), dtype).reshape(shape)

    def free(self):
        self.rt.hipHostFree.argtypes = [ctypes.c_void_p]
        assert self.rt.hipHostFree(self.p) == 0


def test_pinned_arrays_pass_the_stage_by():
    print("[case] host stage use", flush=True)
    n = (127, 127, 127)
    s = plan(n)
    f = np.random.default_rng(1).uniform(-1, 1, n[::-1])
    ans, pin_f, pin_ans = np.empty_like(f), Pinned(f.shape, f.dtype), Pinned(f.shape, f.dtype)
    pin_f.a[:] = f
    s.solve(ans, f)
    want, before = ans.copy(), threads()
    s.solve(pin_ans.a, pin_f.a)
    s.solve(pin_ans.a, pin_f.a)
    assert threads() == before                       # nothing set up for pinned arrays
    assert np.array_equal(pin_ans.a, want)
    s.solve(ans, f)
    workers = threads() - before
    assert len(workers) == 6
    for a, b, used in ((ans, f, True), (pin_ans.a, pin_f.a, False), (ans, pin_f.a, True), (pin_ans.a, f, True)):
        time.sleep(0.05)                             # they spin for 0.2 ms before they sleep
        t = busy(workers)
        a[:] = 0
        s.solve(a, b)
        time.sleep(0.05)
        assert (busy(workers) > t) == used
        assert np.array_equal(a, want)
    del s
    assert not threads() & workers                   # ended with the plan
    pin_f.free()
    pin_ans.free()


@pytest.mark.parametrize("n,staged", [((63, 63, 63), False), ((127, 63, 63), True)])
def test_small_arrays_pass_the_stage_by(n, staged):
    """1.9 MiB, which the runtime copies faster, and 3.8 MiB."""
    print("[case] host stage from", n, flush=True)
    s = plan(n)
    f = np.random.default_rng(1).uniform(-1, 1, n[::-1])
    ans = np.empty_like(f)
    s.solve(ans, f)
    before = threads()
    s.solve(ans, f)
    assert len(threads() - before) == (6 if staged else 0)
