"""Trees and node boxes at the sizes where the 64-leaf grouping of the build can go wrong
(chunk edges, one level more or less, ragged ends), bit for bit against the oracle: the index
tree in closed form (mode 0) and the fitted trees (modes 1, 2), with special coordinates."""
import numpy as np
import pytest

from tests import cases
from tests.test_gpu_parity import _np, _t

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 5, 63, 64, 65, 127, 128, 129, 191, 4095, 4096, 4097, 8192 + 65, 64 * 4096 + 130]


def _check(ccc, oracle, t0, t1, mode):
    ccc.set_morton_mode(mode)
    try:
        bb, tree = ccc.bvh_motion(_t(t0[None]), _t(t1[None]))
    finally:
        ccc.set_morton_mode(0)
    rb, rt, _, _ = oracle.bvh(t0, t1, morton_mode=mode)
    np.testing.assert_array_equal(_np(tree)[0], rt)
    np.testing.assert_array_equal(_np(bb)[0], rb)


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("n", SIZES)
def test_tree_and_boxes(ccc, oracle, n, mode):
    dtype = np.float32 if n % 2 else np.float64
    t0, t1, _ = cases.random_soup(n, seed=n, dtype=dtype)
    _check(ccc, oracle, t0, t1, mode)


def test_clustered_keys(ccc, oracle):
    """Most codes equal: deep fitted trees whose ranges cross chunk edges in every way."""
    t0, t1, _ = cases.random_soup(3000, seed=9)
    t0[:2800] = 0.5 + 1e-9 * t0[:2800]
    t1[:2800] = 0.5 + 1e-9 * t1[:2800]
    for mode in (0, 1, 2):
        _check(ccc, oracle, t0, t1, mode)


def test_special_coordinates(ccc, oracle):
    """NaN coordinates are ignored by the unions, infinities kept, whole-NaN boxes stay NaN."""
    t0, t1, _ = cases.random_soup(700, seed=4)
    t0[3], t1[3] = np.nan, np.nan
    t0[64:130], t1[64:130] = np.nan, np.nan
    t0[200, 1, 2] = np.inf
    t1[201, 0] = -np.inf
    t0[500, 2, 0] = np.nan
    _check(ccc, oracle, t0, t1, 0)
