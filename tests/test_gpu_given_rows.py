"""compute_impulses_from_collisions where the split of its rows over waves changes."""
import numpy as np
import pytest

from tests import cases, test_gpu_pairs
from tests.test_gpu_parity import _np, _t

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("m", [32, 63, 65, 16383, 16384, 16385])
def test_rows_at_the_edges_of_waves(ccc, oracle, m, dtype):
    """Two meshes' rows: 32 per wave up to 32,768 in all, 64 from there on."""
    test_gpu_pairs.test_impulses_of_given_rows(ccc, oracle, m, dtype)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("rows", [(0, 0), (0, 900), (900, 0), (39, 39), (40, 40), (41, 39), (3000, 65536), (-900, -65536)])
def test_long_lists_with_few_and_many_rows(ccc, oracle, rows, dtype):
    """Lists of 65,536 rows on two meshes of 40 triangles, from none to all of them given (negative:
    scattered over the list): summed directly or in lines, as four places of the lists say.  Float
    sums of at most 4 k terms: within 8 k ulp of the largest."""
    n, m = 40, 65536
    c = -np.ones((2, m, 3), np.int64)
    r = np.zeros((2, m, 1), dtype)
    t, want = [], []
    for b in range(2):
        t0, t1, mass = cases.random_soup(n, seed=7 + b, motion=0.2, dtype=dtype)
        rb, rt, _, _ = oracle.bvh(t0, t1)
        coll, roots, _ = oracle.find_collisions_continuous(rb, rt, t0, t1)
        rng = np.random.default_rng(b)
        k = abs(rows[b])
        at = np.arange(k) if rows[b] >= 0 else np.sort(rng.permutation(m)[:k])
        pick = rng.integers(0, len(coll), k)
        c[b][at], r[b, at, 0] = coll[pick], roots[pick]
        t.append((t0, t1, mass))
        want.append(oracle.impulses(t0, t1, mass, coll[pick], roots[pick]) if k else [np.zeros((n, 3, 3)), np.zeros((n, 3, 3)), np.zeros((n, 3), np.int32)])
    t0, t1, mass = (np.stack(x) for x in zip(*t))
    dv, dx, cnt = (_np(x) for x in ccc.compute_impulses_from_collisions(_t(c), _t(r), _t(t0), _t(t1), _t(mass)))
    for b in range(2):
        np.testing.assert_array_equal(cnt[b], want[b][2])
        for got, ref in ((dv[b], want[b][0]), (dx[b], want[b][1])):
            tol = 8 * max(abs(rows[b]), 1) * np.finfo(dtype).eps * max(np.abs(ref).max(), np.finfo(dtype).tiny)
            assert np.abs(got - ref).max() <= tol + 1e-12 * np.abs(ref).max()
