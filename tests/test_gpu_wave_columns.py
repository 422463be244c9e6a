"""Columns of 255 and 511 points, a half or a whole wavefront to each pair (axis_kernels.hip:
yaxis_wave_kernel), at the edges of its 8- and 16-column tiles, against the
oracle: one column, ragged last tiles, and launches on both sides of the line
between the two widths (128 tiles of 16), which give the same bits.

FP64: 1e-12 relative, the bar of every FP64 solve here; FP32: float rounding of
input, transforms and scales, 4e-6; FP32+refine: 1e-9."""
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


@pytest.mark.parametrize("nx", [1, 2, 7, 8, 9, 15, 16, 17, 33, 100])
@pytest.mark.parametrize("ny", [255, 511])
@pytest.mark.parametrize("prec,tol", [("f64", 1e-12), ("f32", 4e-6), ("refine", 1e-9)])
def test_columns(fdm, nx, ny, prec, tol):
    import torch
    print("[case] wave columns", nx, ny, prec, flush=True)
    dx, dy = 2 * np.pi / max(nx, 2), 2 * np.pi / ny
    g = (dx, dy, (nx + 1) * dx, (ny + 1) * dy)
    s = fdm.LaplRect(*g, nx, ny, precision=prec)
    tiles = (nx + 15) // 16
    batch = 128 // tiles + 1                    # 16-column tiles; one problem takes 8
    f = np.stack([O.field(3 + b, (ny, nx)) for b in range(3)]).astype(s.dtype)
    rhs = torch.from_numpy(f[np.arange(batch) % 3]).cuda()
    ans = torch.zeros_like(rhs)
    s.solve_batch(ans, rhs)
    one = torch.zeros_like(rhs[0])
    got = ans.cpu().numpy()
    for b in range(3):
        s.solve(one, rhs[b])
        assert np.array_equal(one.cpu().numpy(), got[b]), b
        assert rel(got[b].astype(np.float64), O.lapl_rect(f[b].astype(np.float64), *g)) <= tol, b
    assert np.array_equal(got[batch - 1], got[(batch - 1) % 3])


@pytest.mark.parametrize("ny", [255, 511])
@pytest.mark.parametrize("prec,tol", [("f64", 1e-12), ("f32", 4e-6)])
def test_planes(fdm, ny, prec, tol):
    """Planes of a cube (15 x ny x 7) through the same tiles, set as a variant."""
    print("[case] wave planes", ny, prec, flush=True)
    n = (15, ny, 7)
    h = [2 * np.pi / v for v in n]
    g = (*h, *[2 * np.pi + v for v in h])
    s = fdm.LaplCube(*g, *n, precision=prec)
    s.variant = next(v for v in s.variants() if v[0] == 0 and v[2] == 16)
    f = O.field(5, (n[2], n[1], n[0])).astype(s.dtype)
    ans = np.empty_like(f)
    s.solve(ans, f)
    assert rel(ans.astype(np.float64), O.lapl_cube(f.astype(np.float64), *g)) <= tol
