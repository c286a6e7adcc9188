"""Simulations on a fitted tree sum their impulses in one line per corner: the same counts as
the index tree's direct sums, and the same sums to rounding."""
import numpy as np
import pytest

from tests.test_gpu_parity import _np, _t
from tests.test_gpu_sim import _scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [5, 9, 18])
@pytest.mark.parametrize("graph", [True, False])
def test_fitted_simulation_sums(ccc, n, dtype, graph):
    """One pass on grids of 32 to 578 triangles, its faces shuffled.  A corner's sum of k shares
    is off by at most k ulp of the sum of their sizes, and the shares are at most the largest
    sum's size times k: 8 k^2 ulp of the largest covers both sides."""
    sc = _scene(n, 7)
    f = sc.faces[np.random.default_rng(n).permutation(len(sc.faces))]
    m = np.random.default_rng(1).uniform(0.5, 2.0, sc.x0.shape[0])[f]
    out = []
    for morton in (0, 1, 2):
        sim = ccc.Sim(_t(sc.x0.astype(dtype)), _t(sc.x1.astype(dtype)), _t(f), _t(m.astype(dtype)), iters=1,
                      max_candidates=512, morton=morton, graph=graph)
        sim.step()
        out.append([_np(a) for a in sim.last_impulses()] + [_np(sim.positions()[1])])
    dv, dx, cnt, x1 = out[0]
    k = max(int(cnt.max()), 1)
    for got in out[1:]:
        np.testing.assert_array_equal(got[2], cnt)
        for a, b in zip((got[0], got[1]), (dv, dx)):
            fin = np.isfinite(b)
            np.testing.assert_array_equal(np.isfinite(a), fin)
            assert np.abs(a[fin] - b[fin]).max() <= 8 * k * k * np.finfo(dtype).eps * np.abs(b[fin]).max()
        far = max(np.abs(x1).max(), np.abs(dx[np.isfinite(dx)]).max())
        assert np.abs(got[3] - x1).max() <= 64 * k * np.finfo(dtype).eps * far
