"""Small cubes in one launch or three (fdmgpu.hip: use_small_cube): which of the two a
solve takes depends on the batch where three launches of few problems are faster, so
both give the same bits: the default variant against the three launches set as a
variant (z systems in the default layout, named)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fdm():
    import fdm_amd
    return fdm_amd


def plan(fdm, n, prec):
    h = [2 * np.pi / m for m in n]
    return fdm.LaplCube(*h, *[2 * np.pi + v for v in h], *n, precision=prec)


@pytest.mark.parametrize("nz", [15, 31])
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_same_bits(fdm, nz, prec):
    import torch
    print("[case] small cube route", nz, prec, flush=True)
    s = plan(fdm, (15, 15, nz), prec)
    default = s.variant
    f = torch.from_numpy(np.random.default_rng(1).uniform(-1, 1, (64, nz, 15, 15)).astype(s.dtype)).cuda()
    for batch in (1, 47, 48, 64):
        got, want = torch.zeros_like(f[:batch]), torch.zeros_like(f[:batch])
        s.variant = default
        s.solve_batch(got, f[:batch].contiguous())
        s.variant = (1, 0, 0, 5, 0)
        s.solve_batch(want, f[:batch].contiguous())
        assert torch.equal(got, want), batch


@pytest.mark.parametrize("nz,prec,batch,one", [(31, "f64", 1, False), (31, "f64", 47, False), (31, "f64", 48, True),
                                               (31, "f32", 1, True), (15, "f64", 1, True), (15, "f32", 1, True)])
def test_route(fdm, nz, prec, batch, one):
    from fdm_amd import hip
    print("[case] small cube launches", nz, prec, batch, flush=True)
    s = plan(fdm, (15, 15, nz), prec)
    rhs, ans = (hip.DeviceArray.from_host(np.ones((batch, nz, 15, 15), s.dtype)) for _ in range(2))
    s.set_timing()
    s.solve_batch(ans, rhs)
    assert {k: n for k, (_, n) in s.timing().items()} == ({"other": 1} if one else {"xy_fwd": 1, "zcr": 1, "xy_inv": 1})
