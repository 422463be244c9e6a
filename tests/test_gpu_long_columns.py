"""z systems of 511 rows of floats, eliminated in double with one lane to 64 rows by
default (cr_kernels.hip), against the oracle's FP64 solve and the other layouts set as
variants.  Float rounding of input, transforms and answer, 4e-6; between layouts, which
differ only in the rounding of the double elimination, one rounding of the answer,
6e-8, through two transforms whose float rounding it may flip: 1e-6."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm((a - b).ravel()) / np.linalg.norm(b.ravel()))


@pytest.mark.parametrize("n", [(3, 7, 511), (15, 15, 511), (63, 31, 511)])
def test_columns_of_511(n):
    import fdm_amd
    print("[case] long columns", n, flush=True)
    h = [2 * np.pi / v for v in n]
    g = (*h, *[2 * np.pi + v for v in h])
    s = fdm_amd.LaplCube(*g, *n, precision="f32")
    f = O.field(3, n[::-1]).astype(np.float32)
    ans, other = np.empty_like(f), np.empty_like(f)
    s.solve(ans, f)
    assert rel(ans.astype(np.float64), O.lapl_cube(f.astype(np.float64), *g)) <= 4e-6
    for v in s.variants():
        if v[0] == 1 and v[3]:
            s.variant = v
            s.solve(other, f)
            assert rel(other.astype(np.float64), ans.astype(np.float64)) <= 1e-6, v
