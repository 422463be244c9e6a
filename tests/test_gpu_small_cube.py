"""Cubes of 15 x 15 x 15 and 15 x 15 x 31 points solved by one block each
(small_kernels.hip), against the oracle and against the three-launch path (the
variant that names the z kernel): single, batched, in place, through a pointer
table with a right-hand side apart.

FP64: 1e-12 relative, the bar of every FP64 solve here; FP32: float rounding of
input, transforms and eigenvalues, 4e-6."""
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


@pytest.mark.parametrize("n", [(15, 15, 15), (15, 15, 31)])
@pytest.mark.parametrize("prec,tol", [("f64", 1e-12), ("f32", 4e-6)])
def test_small(fdm, n, prec, tol):
    import torch
    print("[case] small cube", n, prec, flush=True)
    h = (2 * np.pi / n[0], 2 * np.pi / n[1], 3.0 / n[2])
    g = (*h, *[(v + 1) * a for v, a in zip(n, h)])
    s = fdm.LaplCube(*g, *n, precision=prec)
    old = fdm.LaplCube(*g, *n, precision=prec)
    old.variant = next(v for v in old.variants() if v[0] == 1 and v[3] != 0)
    f = np.stack([O.field(9 + k, n[::-1]) for k in range(3)]).astype(s.dtype)
    rhs = torch.from_numpy(f).cuda()
    ans = torch.full_like(rhs, 7)
    s.solve_batch(ans, rhs)
    assert np.array_equal(rhs.cpu().numpy(), f)
    ref = torch.zeros_like(rhs)
    old.solve_batch(ref, rhs)
    one = rhs[1].clone()
    s.solve(one, one)                                       # in place
    host = np.empty_like(f[2])
    s.solve(host, f[2])
    got = ans.cpu().numpy()
    assert np.array_equal(one.cpu().numpy(), got[1]) and np.array_equal(host, got[2])
    for k in range(3):
        assert rel(got[k].astype(np.float64), O.lapl_cube(f[k].astype(np.float64), *g)) <= tol, k
    assert rel(got.astype(np.float64), ref.cpu().numpy().astype(np.float64)) <= tol
