"""Static queries on lists long enough for several items per thread: rows against the oracle,
and at an output that does not hold them all."""
import numpy as np
import pytest

from tests import cases
from tests.conftest import sorted_rows, valid_rows
from tests.test_gpu_parity import _np, _t

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("query", ["find_proximity", "find_collisions"])
def test_long_lists(ccc, oracle, query, dtype):
    t, _, _ = cases.random_soup(7000, seed=1, dtype=dtype)
    rb, rt, _, _ = oracle.bvh(t)
    ref = getattr(oracle, query)(rb, rt, t, 2e-3)
    ref = ref[0] if query == "find_proximity" else ref
    want = sorted_rows(ref)
    args = (_t(rb[None]), _t(rt[None]), _t(t[None]), 2e-3)
    got = valid_rows(_np(getattr(ccc, query)(*args, 64)[0]))
    k, m = ccc.last_counts()[0][:2]
    assert (m if query == "find_proximity" else k) > 131072      # the several-items branch
    np.testing.assert_array_equal(sorted_rows(got), want)
    # one row per triangle: a full output, every row one of the oracle's and none twice
    with pytest.warns(UserWarning):
        part = valid_rows(_np(getattr(ccc, query)(*args, 1)[0]))
    if len(want) > 7000:
        assert len(part) == 7000
    part = {tuple(r) for r in part.tolist()}
    assert len(part) == min(7000, len(want)) and part <= {tuple(r) for r in want.tolist()}
