"""The pivoting row elimination of FP32+refine plans holds its four arrays of floats
in LDS: two rows of 4000 points to a CU at a time (64 KB each of 160).

One lane of a block works, so a launch takes one row's time for every round of
blocks: 127 rows are one round on 256 CUs, 8 problems of them (1016 blocks) two
with two blocks a CU and four with one.  Between the two lies 3."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_two_rows_to_a_cu():
    import fdm_amd
    from fdm_amd import hip
    print("[case] pivoted rows in LDS", flush=True)
    nx, ny = 4000, 127
    dx, dy = 2 * np.pi / nx, 2 * np.pi / ny
    s = fdm_amd.LaplRect(dx, dy, (nx + 1) * dx, (ny + 1) * dy, nx, ny, precision="refine")
    s.set_scales(L_scale=np.full(nx + 1, 1.3), U_scale=np.full(nx + 1, 1.1))
    s.set_refine(1e-10, 1)
    t = {}
    for batch in (1, 8):
        rhs, ans = (hip.DeviceArray.from_host(np.ones((batch, ny, nx))) for _ in range(2))
        s.solve_batch(ans, rhs)
        s.set_timing(kernels=["rowcr"])
        for _ in range(3):
            s.solve_batch(ans, rhs)
        ms, n = s.timing()["rowcr"]
        s.set_timing(False)
        t[batch] = ms / n
    print("[time] %.2f ms, %.2f ms" % (t[1], t[8]), flush=True)
    assert t[8] < 3 * t[1]
