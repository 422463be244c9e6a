"""FP32 planes of N = 256 held in registers (plane_reg_kernels.hip): the default
variant takes that kernel when a launch has at least 192 planes and the axis
tiles otherwise, and both give the same bits -- so does the tile variant pinned
at its default sizes.  Every input / output form: FP32, FP32 + FP64 refinement
with problems that converge after different numbers of inner solves, in place,
periodic.

Tolerance of the FP32 solves against the FP64 oracle: four length-256 transforms
in float, each with an error of about eps sqrt(log2 N) = 2e-7, and eigenvalues
rounded to float (6e-8): 5e-6 leaves a factor of five."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

TILES = (0, 32, 64)   # the tile sizes that 0 stands for


@pytest.fixture(scope="module")
def fdm():
    import fdm_amd
    return fdm_amd


def geometry(n, periodic=False):
    h = [2 * np.pi / m for m in n]
    return h + [2 * np.pi + (0 if periodic else v) for v in h]


def rel(a, b):
    return float(np.linalg.norm((a - b).ravel()) / np.linalg.norm(b.ravel()))


def tiles_like_default(s, q):
    zcr = 3 if q >= 8 else 5   # the default z solve of 2^q - 1 rows
    return next(v for v in s.variants() if v[:3] == TILES and v[3] == (zcr if q > 3 else 1))


# planes a launch: 3 x 1, 2 x 95 (tiles), 3 x 64, 1 x 255 (registers)
@pytest.mark.parametrize("nz,batch", [(1, 3), (63, 4), (127, 1), (127, 2), (255, 1)])
def test_f32_planes(fdm, nz, batch):
    from fdm_amd import hip
    print("[case] register planes f32", nz, batch, flush=True)
    n = (255, 255, nz)
    g = geometry(n)
    f = O.field(3, n[::-1]).astype(np.float32)
    s = fdm.LaplCube(*g, *n, precision="f32")
    assert s.variant == (0, 0, 0, 0, 0)
    stack = np.stack([f, f[:, ::-1].copy(), -f, 2 * f][:batch])
    rhs, ans = hip.DeviceArray.from_host(stack), hip.DeviceArray(stack.shape, np.float32)
    s.solve_batch(ans, rhs)
    got = ans.download()
    one = np.empty_like(f)
    for k in range(batch):   # alone: below 192 planes the tiles
        s.solve(one, np.ascontiguousarray(stack[k]))
        assert np.array_equal(got[k], one)
    s.solve_batch(rhs, rhs)   # in place
    assert np.array_equal(got, rhs.download())
    want = O.lapl_cube(f.astype(np.float64), *g)
    assert rel(got[0], want) <= 5e-6
    s.variant = tiles_like_default(s, int(np.log2(nz + 1)))
    s.solve(one, f)
    assert np.array_equal(got[0], one)


@pytest.mark.parametrize("nz", [2, 64, 256])
def test_periodic_f32_planes(fdm, nz):
    from fdm_amd import hip
    print("[case] register planes periodic f32", nz, flush=True)
    n = (256, 256, nz)
    g = geometry(n, True)
    f = O.field(3, n[::-1]).astype(np.float32)
    s = fdm.LaplCube(*g, *n, precision="f32", periodic=True)
    count = max(1, -(-192 // nz))
    stack = np.stack([f] + [f[::-1].copy()] * (count - 1))
    rhs, ans = hip.DeviceArray.from_host(stack), hip.DeviceArray(stack.shape, np.float32)
    s.solve_batch(ans, rhs)
    got = ans.download()
    want = O.lapl_cube(f.astype(np.float64), *g, periodic=True)
    assert rel(got[0], want) <= 5e-6
    s.variant = next(v for v in s.variants() if v[:3] == TILES and v[3] == (2 if nz >= 64 else 1))
    one = np.empty_like(f)
    s.solve(one, f)
    assert np.array_equal(got[0], one)


@pytest.mark.parametrize("nz", [3, 63, 127])
def test_refine_planes_mixed_batch(fdm, nz):
    from fdm_amd import hip
    print("[case] register planes refine", nz, flush=True)
    n = (255, 255, nz)
    g = geometry(n)
    shape = n[::-1]
    x = [np.sin(np.pi * np.arange(1, m + 1) / (m + 1)) for m in shape]
    smooth = x[0][:, None, None] * x[1][None, :, None] * x[2][None, None, :]   # needs more inner solves
    stack = np.stack([O.field(4, shape), np.zeros(shape), smooth, O.field(5, shape)])
    s = fdm.LaplCube(*g, *n, precision="refine")
    rhs, ans = hip.DeviceArray.from_host(stack), hip.DeviceArray(stack.shape, np.float64)
    s.solve_batch(ans, rhs)
    got = ans.download()
    assert s.stats().max_rel_residual <= 1e-10
    for k in range(len(stack)):
        a1, r1 = hip.DeviceArray(shape, np.float64), hip.DeviceArray.from_host(stack[k])
        s.solve(a1, r1)
        assert np.array_equal(a1.download(), got[k])
        if stack[k].any():
            assert rel(got[k], O.lapl_cube(stack[k], *g)) <= 1e-9
    default = s.variant
    s.variant = tiles_like_default(s, int(np.log2(nz + 1)))
    s.solve_batch(ans, rhs)
    assert np.array_equal(ans.download(), got)
    s.variant = default
    s.solve_batch(rhs, rhs)   # in place
    assert np.array_equal(rhs.download(), got)
