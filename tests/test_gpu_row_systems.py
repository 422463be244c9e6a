"""LaplRect's row systems, one wavefront per row (cr_kernels.hip: rowpart_kernel),
at the edges of its chunk sizes (64 lanes of 1, 2, 4, 8, 16 unknowns; beyond 1024
points the LDS kernel), with unit scales and with scales, against the oracle's
gtsv.

FP64: 1e-12 relative, the bar of every FP64 solve here.  FP32 data (elimination
in FP64): float rounding of input, transforms and scales, 2e-6, times the
conditioning of a random right-hand side, of order one."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fdm():
    import fdm_amd
    return fdm_amd


def rel(a, b):
    return float(np.linalg.norm((a - b).ravel()) / np.linalg.norm(b.ravel()))


@pytest.mark.parametrize("nx", [1, 2, 3, 63, 64, 65, 127, 128, 129, 255, 257, 511, 512, 513, 1000, 1024, 1025])
@pytest.mark.parametrize("scaled", [False, True])
def test_rows(fdm, nx, scaled):
    print("[case] row systems", nx, scaled, flush=True)
    ny = 15
    dx, dy = 2 * np.pi / max(nx, 2), 2 * np.pi / ny
    g = (dx, dy, (nx + 1) * dx, (ny + 1) * dy)
    f = O.field(7, (ny, nx))
    sc = {}
    if scaled:
        r = np.linspace(1.0, 2.0, nx + 1)
        sc = {"lm_y_scale": 1 / r ** 2, "L_scale": 1 - 0.25 / (nx + r), "U_scale": 1 - 0.5 / (nx + r)}
    for prec, tol in (("f64", 1e-12), ("f32", 4e-6)):
        s = fdm.LaplRect(*g, nx, ny, precision=prec)
        if scaled:
            s.set_scales(**sc)
        rhs = f.astype(s.dtype)
        ans = np.empty_like(rhs)
        s.solve(ans, rhs)
        # the matrix of a float plan is that of its scales rounded to float
        own = {k: v.astype(s.dtype).astype(np.float64) for k, v in sc.items()}
        assert rel(ans, O.lapl_rect(rhs.astype(np.float64), *g, **own)) <= tol, prec
