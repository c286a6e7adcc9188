"""Stateless queries in a context that fits its trees: they walk the tree at once."""
import numpy as np
import pytest

from tests import cases
from tests.conftest import sorted_rows, valid_rows
from tests.test_gpu_parity import _np, _t
from tests.test_zz_no_alloc import _call, _compare, capi  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [1, 2, 64, 700])
def test_nothing_is_prepared_for_the_other_path(ccc, oracle, n, dtype):
    """One preparation (the walk's) per static query, two with the moving vertices' records; the
    results equal the index tree's."""
    t0, t1, m = cases.random_soup(n, seed=n + 2, motion=0.2, dtype=dtype)
    a0, a1, am = (_t(a[None]) for a in (t0, t1, m))
    bb, tree = ccc.bvh(a0)
    mb, mt = ccc.bvh_motion(a0, a1)
    want = [_np(ccc.find_collisions(bb, tree, a0, 1e-3, 64)), _np(ccc.compute_impulses(mb, mt, a0, a1, am, n, 16)[2])]
    ccc.set_morton_mode(1)
    try:
        bb, tree = ccc.bvh(a0)
        mb, mt = ccc.bvh_motion(a0, a1)
        prepared = []
        got = []
        for call in (lambda: ccc.find_collisions(bb, tree, a0, 1e-3, 64), lambda: ccc.compute_impulses(mb, mt, a0, a1, am, n, 16)[2]):
            ccc.set_profiling(True)
            got.append(_np(call()))
            prepared.append(ccc.kernel_times()["tree_prep"][1])
            ccc.set_profiling(False)
    finally:
        ccc.set_profiling(False)
        ccc.set_morton_mode(0)
    assert prepared == [1, 2]
    np.testing.assert_array_equal(sorted_rows(valid_rows(got[0][0])), sorted_rows(valid_rows(want[0][0])))
    np.testing.assert_array_equal(got[1], want[1])


@pytest.mark.parametrize("maxc", [1, 300])
def test_allocation_free_call(ccc, capi, maxc):  # noqa: F811
    """The scratch array holds the walk's buffers at once; with one candidate per triangle the
    list grows and they are made again behind it."""
    import ctypes
    lib, ctx, plain, noalloc = capi
    lib.ccc_context_set_morton.argtypes = [ctypes.c_void_p, ctypes.c_int]
    t0, t1, m = cases.folded(20, seed=2)
    args = [_t(a[None]) for a in (t0, t1, m)]
    bb, tree = ccc.bvh_motion(args[0], args[1])
    ref = _call(capi, plain, bb, tree, *args, 300)
    assert lib.ccc_context_set_morton(ctx, 1) == 0
    try:
        for fn in (plain, noalloc):
            st, *rest = _call(capi, fn, bb, tree, *args, maxc)
            assert bool(st & 0x100) == (maxc == 1)
            _compare(ref, (st & 0xff, *rest))
    finally:
        assert lib.ccc_context_set_morton(ctx, 0) == 0
