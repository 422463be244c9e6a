"""The convergence check inside the residual launch (refine.hip): the reported
residual against one computed on the host, and a batch whose problems converge
after different numbers of inner solves against the same problems alone.

Tolerance of the reported residual: the device and the host both compute
||f - A u|| / ||f|| in FP64; each element's rounding is a few eps ||A|| |u|,
eps ||A|| ||u|| / ||f|| <= 2.2e-16 * 12 / h^2 * (h^2 N^2 / pi^2) / 3 ~ 1e-11 at
N = 256 for the smoothest f, so 2e-11 absolute plus 1e-9 relative."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fdm():
    import fdm_amd
    return fdm_amd


def smooth(shape):
    out = 1.0
    for n in shape:
        out = np.multiply.outer(out, np.sin(np.pi * np.arange(1, n + 1) / (n + 1)))
    return out


def solver(fdm, shape):
    n = shape[::-1]
    h = [2 * np.pi / max(shape)] * len(n)
    l = [(m + 1) * v for m, v in zip(n, h)]
    cls = fdm.LaplCube if len(n) == 3 else fdm.LaplRect
    return cls(*h, *l, *n, precision="refine"), h


# granule, chunk and tile edges: one plane, a granule of 8 planes and one more,
# several tiles with a ragged last one, 32 granules in one chunk; 2-D rows
@pytest.mark.parametrize("shape", [(1, 3, 3), (7, 7, 7), (15, 31, 63), (63, 127, 31), (127, 15, 255), (255, 7, 127),
                                   (255, 255, 255), (3, 5), (127, 100), (511, 1000)])
@pytest.mark.parametrize("iters", [1, 4])
def test_residual_and_mixed_batch(fdm, shape, iters):
    from fdm_amd import hip
    print("[case] folded check", shape, iters, flush=True)
    s, h = solver(fdm, shape)
    s.set_refine(1e-10, iters)
    fields = [np.zeros(shape), O.field(5, shape), smooth(shape), O.field(6, shape)]   # zero f: done at once
    if np.prod(shape) > 2 ** 22:
        fields = fields[:2]
    batch = np.stack(fields)
    rhs, ans = hip.DeviceArray.from_host(batch), hip.DeviceArray(batch.shape, np.float64)
    s.solve_batch(ans, rhs)
    st, got = s.stats(), ans.download()
    worst, most = 0.0, 0
    for k, f in enumerate(fields):
        r1, a1 = hip.DeviceArray.from_host(f), hip.DeviceArray(shape, np.float64)
        s.solve(a1, r1)
        one, u = s.stats(), a1.download()
        assert np.array_equal(u, got[k])
        want = O.rel_residual(f, u, *h) if f.any() else 0.0
        assert abs(one.rel_residual - want) <= 2e-11 + 1e-9 * want
        assert one.iterations <= iters and (iters == 1 or one.rel_residual <= 1e-10)
        worst, most = max(worst, one.rel_residual), max(most, one.iterations)
    assert st.max_rel_residual == worst and st.iterations == most
