"""Host-array solves through pinned memory (host_stage.hip): bitwise the device
solve of the same field, on a plan's first call (the runtime's copies), later
calls (the stage), at sizes around its pieces (512 KiB), groups (1, 2, 4, 8, 16
MiB) and halves (16 MiB, three of them in the largest), from two threads at once
and after every plan that held the stage is gone."""
import threading

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fdm():
    import fdm_amd
    return fdm_amd


def plan(fdm, n, precision):
    h = [2 * np.pi / m for m in n]
    return fdm.LaplCube(*h, *[(m + 1) * v for m, v in zip(n, h)], *n, precision=precision)


def device_answer(s, f):
    from fdm_amd import hip
    rhs, ans = hip.DeviceArray.from_host(f), hip.DeviceArray(f.shape, f.dtype)
    s.solve(ans, rhs)
    hip.synchronize()
    return ans.download()


# (127, 127, 15) FP64 1.8 MiB, FP32 0.9 (below the stage); 3.8, 15.6, 31.4, 62.9 MiB in FP64
@pytest.mark.parametrize("n", [(127, 127, 15), (127, 63, 63), (127, 127, 127), (127, 127, 255), (255, 127, 255)])
@pytest.mark.parametrize("precision", ["f64", "f32", "refine"])
def test_host_solve_is_the_device_solve(fdm, n, precision):
    print("[case] host stage", n, precision, flush=True)
    s = plan(fdm, n, precision)
    want, ans = {}, np.empty(n[::-1], s.dtype)
    for k in range(4):
        f = O.field(10 + k % 2, n[::-1]).astype(s.dtype)
        if k < 2:
            want[k] = device_answer(s, f)
        ans[:] = np.nan
        s.solve(ans, f)
        assert np.array_equal(ans, want[k % 2]), k
    s.solve(f, f)   # in place
    assert np.array_equal(f, want[1])


def test_two_threads(fdm):
    n = (127, 127, 63)
    fields = [O.field(3, n[::-1]), O.field(4, n[::-1])]
    want = [device_answer(plan(fdm, n, "f64"), f) for f in fields]
    bad = []

    def run(i):
        s, ans = plan(fdm, n, "f64"), np.empty(n[::-1])
        for _ in range(12):
            ans[:] = np.nan
            s.solve(ans, fields[i])
            if not np.array_equal(ans, want[i]):
                bad.append(i)

    ts = [threading.Thread(target=run, args=(i,)) for i in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
