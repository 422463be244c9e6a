"""LaplRect and LaplCyl3FFT2 rows of more than 1024 points (cr_kernels.hip:
rowcr_kernel), at the edges of its levels and of its two block sizes (three rows of
1706 points fit a CU's LDS, of 1707 two), with unit scales and with scales, against
the oracle's gtsv.

The spacings keep the systems well conditioned (about 100), so that the oracle's own
elimination is good to 1e-13: FP64 1e-12 relative, the bar of every FP64 solve
here; FP32 data float rounding of input, transforms and scales, 4e-6;
FP32+refine 1e-9."""
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


@pytest.mark.parametrize("nx", [1025, 1536, 1706, 1707, 2047, 2048, 2049, 3000, 4095, 4096])
@pytest.mark.parametrize("scaled", [False, True])
def test_long_rows(fdm, nx, scaled):
    import torch
    print("[case] long rows", nx, scaled, flush=True)
    ny, dx = 15, 0.5
    dy = 2 * np.pi / ny
    g = (dx, dy, (nx + 1) * dx, (ny + 1) * dy)
    f = np.stack([O.field(7 + b, (ny, nx)) for b in range(2)])
    sc = {}
    if scaled:
        r = np.linspace(1.0, 2.0, nx + 1)
        sc = {"lm_y_scale": 1 / r ** 2, "L_scale": 1 - 0.25 / (nx + r), "U_scale": 1 - 0.5 / (nx + r)}
    for prec, tol in (("f64", 1e-12), ("f32", 4e-6), ("refine", 1e-9)):
        s = fdm.LaplRect(*g, nx, ny, precision=prec)
        if scaled:
            s.set_scales(**sc)
        rhs = torch.from_numpy(f.astype(s.dtype)).cuda()
        ans = torch.zeros_like(rhs)
        s.solve_batch(ans, rhs)
        # the matrix of a float plan is that of its scales rounded to float
        own = {k: v.astype(s.dtype).astype(np.float64) for k, v in sc.items()}
        for b in range(2):
            want = O.lapl_rect(f[b].astype(s.dtype).astype(np.float64), *g, **own)
            assert rel(ans[b].cpu().numpy().astype(np.float64), want) <= tol, (prec, b)


@pytest.mark.parametrize("nr", [1025, 1706, 1707, 4096])
def test_long_radii(fdm, nr):
    print("[case] long radii", nr, flush=True)
    nz, nphi, dr, r0 = 7, 4, 0.5, 1.0
    dz = 2 * np.pi / nz
    s = fdm.LaplCyl3FFT2(dr, dz, r0, r0 + (nr + 1) * dr, (nz + 1) * dz, nr, nz, nphi)
    f = O.field(9, (nphi, nz, nr))
    ans = np.empty_like(f)
    s.solve(ans, f)
    assert rel(ans, O.lapl_cyl3_fft2(f, dr, dz, r0, (nz + 1) * dz)) <= 1e-12
