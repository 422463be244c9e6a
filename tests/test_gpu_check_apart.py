"""The convergence check as a launch of its own (refine.hip), on both sides of the
lines where the residual launch takes it over: 3-D launches of more than 1024 blocks,
2-D ones of more than 200, or 64 where a problem has more than 32; and the check after
the fourth inner solve, which it takes whatever its size (1e-16 is not reached: every
check finds the problems unfinished).  Problems that converge at once (f = 0) and after different
numbers of inner solves, against the same problems alone, whose launch checks itself:
bitwise the same answers, and the statistics of the worst of them."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def solver(n):
    import fdm_amd
    h = [2 * np.pi / m for m in n]
    cls = fdm_amd.LaplCube if len(n) == 3 else fdm_amd.LaplRect
    return cls(*h, *[(m + 1) * v for m, v in zip(n, h)], *n, precision="refine")


# blocks a problem: a 15 x 15 x 7 cube 1, 31 x 31 x 31 1 to 4 (fewer in larger batches),
# 127 x 31 x 15 4 or 8; 33 x 15 points 8, 100 x 127 32, 20 x 255 64, 9 x 511 128
@pytest.mark.parametrize("n,batches", [((15, 15, 7), (1024, 1025)), ((31, 31, 31), (250, 1030)),
                                       ((127, 31, 15), (256, 300)), ((33, 15), (25, 26)), ((100, 127), (6, 7, 40)),
                                       ((20, 255), (1, 2, 17)), ((9, 511), (1, 9))])
@pytest.mark.parametrize("tol,iters", [(1e-10, 1), (1e-10, 4), (1e-16, 5)])
def test_batch_is_the_problems_alone(n, batches, tol, iters):
    import torch
    print("[case] check apart", n, batches, tol, iters, flush=True)
    s = solver(n)
    s.set_refine(tol, iters)
    shape = n[::-1]
    smooth = 1.0
    for m in shape:
        smooth = np.multiply.outer(smooth, np.sin(np.pi * np.arange(1, m + 1) / (m + 1)))
    fields = np.stack([O.field(5, shape), np.zeros(shape), smooth, 1e6 * O.field(6, shape)])
    alone, stats = [], []
    one = torch.zeros(shape, dtype=torch.float64, device="cuda")
    for f in fields:
        s.solve(one, torch.from_numpy(f).cuda())
        stats.append(s.stats())
        alone.append(one.cpu().numpy())
    for batch in batches:
        rhs = torch.from_numpy(fields[np.arange(batch) % 4]).cuda()
        ans = torch.zeros_like(rhs)
        s.solve_batch(ans, rhs)
        got, st = ans.cpu().numpy(), s.stats()
        for k in range(batch):
            assert np.array_equal(got[k], alone[k % 4]), (batch, k)
        mine = stats[:batch]   # of the fields in this batch
        assert st.iterations == max(v.iterations for v in mine)
        assert st.max_rel_residual == max(v.rel_residual for v in mine)
        assert st.rel_residual == stats[(batch - 1) % 4].rel_residual
