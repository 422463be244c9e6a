"""What is created and destroyed without an error leaves none behind: the caller's
next check of the runtime's last error (torch's, after each of its calls) is clean."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graph", [False, True])
def test_group_leaves_no_error(graph):
    import fdm_amd
    from fdm_amd import hip, serve
    print("[case] group end", graph, flush=True)
    n = 15
    h, l = 2 * np.pi / n, 2 * np.pi + 2 * np.pi / n
    rhs, ans = hip.DeviceArray.from_host(np.ones((n, n, n))), hip.DeviceArray((n, n, n), np.float64)
    p = serve.cube_problem(h, h, h, l, l, l, n, n, n, ans.ptr.value, rhs.ptr.value, precision=fdm_amd.F64)
    hip.rt().hipGetLastError()
    g = serve.Group([p], graph=graph)
    g.solve()
    g.solve()
    hip.synchronize()
    assert hip.rt().hipGetLastError() == 0
    g.close()
    assert hip.rt().hipGetLastError() == 0
