"""Candidate pairs by chunks of 64 leaf positions, at chunk edges and ragged ends: against the
oracle's traversal, and against the general tree walk, which the same boxes take when the
tree's internal rows are numbered differently (the pair sets must be equal)."""
import numpy as np
import pytest

from tests import cases
from tests.conftest import sorted_rows, valid_rows
from tests.test_gpu_parity import _check_close, _compare_collisions, _np, _renumbered_internal_tree, _t

pytestmark = pytest.mark.gpu


def _mincol(ccc, bb, tree, t0, t1, cap):
    out = _np(ccc.find_mincol_cand(_t(bb[None]), _t(tree[None]), _t(t0[None]), _t(t1[None]), cap))[0]
    return sorted_rows(valid_rows(out)), ccc.last_counts()[0][0]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [2, 3, 63, 64, 65, 127, 129, 200, 1000, 4097])
def test_pairs_at_chunk_edges(ccc, oracle, n, dtype):
    t0, t1, _ = cases.random_soup(n, seed=n + 1, dtype=dtype)
    rb, rt, _, _ = oracle.bvh(t0, t1)
    pairs, total = oracle.traverse(rb, rt, 0.0)
    want = sorted_rows(oracle.mincol(t0, t1, pairs))
    cap = total // n + 2
    rows, k = _mincol(ccc, rb, rt, t0, t1, cap)
    assert k == total
    np.testing.assert_array_equal(rows, want)
    if n > 3:
        rows, k = _mincol(ccc, *_renumbered_internal_tree(rb, rt, 2), t0, t1, cap)
        assert k == total
        np.testing.assert_array_equal(rows, want)


@pytest.mark.parametrize("n", [65, 300])
def test_partial_pairs(ccc, oracle, n):
    t0, t1, _ = cases.random_soup(n, seed=n)
    rb, rt, _, _ = oracle.bvh(t0, t1)
    for share in (0.0, 0.03, 0.5, 1.0):
        check = np.random.default_rng(7).random(n) < share
        total = len(oracle.traverse_partial(rb, rt, check))
        counts = []
        for bb, tree in ((rb, rt), _renumbered_internal_tree(rb, rt, 3)):
            ccc.find_collisions_continuous_partial(_t(bb[None]), _t(tree[None]), _t(t0[None]), _t(t1[None]), _t(check[None]), 400, 400)
            counts.append(ccc.last_counts()[0])
        assert counts[0] == counts[1] and counts[0][0] == total


def test_pairs_with_super_boxes(ccc, oracle):
    """More than 4,096 chunks: groups of 64 chunks are tested first."""
    n = 64 * 4096 + 77
    rng = np.random.default_rng(3)
    c = rng.random((n, 1, 3))
    c = c[np.argsort(np.floor(c[:, 0, 0] * 40) * 1000 + c[:, 0, 1])]
    t0 = c + 0.004 * rng.standard_normal((n, 3, 3))
    t1 = t0 + 0.002 * rng.standard_normal((n, 3, 3))
    rb, rt, _, _ = oracle.bvh(t0, t1)
    pairs, total = oracle.traverse(rb, rt, 0.0)
    assert total > n // 4
    rows, k = _mincol(ccc, rb, rt, t0, t1, total // n + 2)
    assert k == total
    np.testing.assert_array_equal(rows, sorted_rows(oracle.mincol(t0, t1, pairs)))


def test_special_boxes(ccc, oracle):
    """NaN triangles meet nothing; infinite ones meet everything on their axis."""
    t0, t1, _ = cases.random_soup(200, seed=8)
    t0[5], t1[5] = np.nan, np.nan
    t0[64:128, :, 1], t1[64:128, :, 1] = np.nan, np.nan
    t0[150, 0] = np.inf
    t1[151, 1] = -np.inf
    rb, rt, _, _ = oracle.bvh(t0, t1)
    _, total = oracle.traverse(rb, rt, 0.0)
    for bb, tree in ((rb, rt), _renumbered_internal_tree(rb, rt, 2)):
        _, k = _mincol(ccc, bb, tree, t0, t1, 200)
        assert k == total


@pytest.mark.parametrize("chunk", [0, 1, 64, 65, 1000])
@pytest.mark.parametrize("n", [2, 9, 70, 300])
def test_items_at_batch_edges(ccc, oracle, n, chunk):
    """The narrow phase's items in waves of 64 pairs and chunks of them: collisions, counts and
    the two ways to impulses against the oracle."""
    t0, t1, m = cases.random_soup(n, seed=n + 5, motion=0.2)
    rb, rt, _, _ = oracle.bvh(t0, t1)
    dv, dx, cnt, coll, roots, counts = oracle.compute_impulses(rb, rt, t0, t1, m)
    args = (_t(rb[None]), _t(rt[None]), _t(t0[None]), _t(t1[None]))
    want = [counts[k] for k in ("candidates", "subprims", "roots", "collisions")]
    ccc.set_pair_chunk(chunk)
    try:
        gc, gr = ccc.find_collisions_continuous(*args, n, 4 * n)
        assert ccc.last_counts()[0] == want
        _compare_collisions(_np(gc)[0], _np(gr)[0], coll, roots)
        direct = ccc.compute_impulses(*args, _t(m[None]), n, 16)
        assert ccc.last_counts()[0] == want
    finally:
        ccc.set_pair_chunk(0)
    for out in (direct, ccc.compute_impulses_from_collisions(gc, gr, args[2], args[3], _t(m[None]))):
        np.testing.assert_array_equal(_np(out[2])[0], cnt)
        _check_close(_np(out[0])[0], dv, "dv")
        _check_close(_np(out[1])[0], dx, "dx")


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("m", [1, 31, 33, 64, 127, 129, 300, 32767, 32768])
def test_impulses_of_given_rows(ccc, oracle, m, dtype):
    """compute_impulses_from_collisions at the edges of its runs: two meshes' rows with padding
    and out-of-range rows among them, shuffled, each row more than once, so that one corner
    takes many shares; from 65,536 rows on they are summed in lines.  Float sums of at most 4 m terms: within 8 m ulp of the largest."""
    c = -np.ones((2, m, 3), np.int64)
    r = np.zeros((2, m, 1), dtype)
    t, want = [], []
    for b in range(2):
        t0, t1, mass = cases.random_soup(40, seed=3 * m + b, motion=0.2, dtype=dtype)
        rb, rt, _, _ = oracle.bvh(t0, t1)
        coll, roots, _ = oracle.find_collisions_continuous(rb, rt, t0, t1)
        rng = np.random.default_rng(m + b)
        pick = rng.integers(0, len(coll), m)
        c[b], r[b, :, 0] = coll[pick], roots[pick]
        keep = rng.random(m) < 0.8
        c[b][~keep] = rng.permutation(np.array([[-1, -1, -1], [40, 0, 0], [0, 40, 3], [0, 1, 15], [1, -5, 2]]))[rng.integers(0, 5, (~keep).sum())]
        t.append((t0, t1, mass))
        want.append(oracle.impulses(t0, t1, mass, c[b][keep], r[b, keep, 0]))
    t0, t1, mass = (np.stack(x) for x in zip(*t))
    dv, dx, cnt = (_np(x) for x in ccc.compute_impulses_from_collisions(_t(c), _t(r), _t(t0), _t(t1), _t(mass)))
    for b in range(2):
        np.testing.assert_array_equal(cnt[b], want[b][2])
        for got, ref in ((dv[b], want[b][0]), (dx[b], want[b][1])):
            tol = 8 * m * np.finfo(dtype).eps * max(np.abs(ref).max(), np.finfo(dtype).tiny)
            assert np.abs(got - ref).max() <= tol + 1e-12 * np.abs(ref).max()


@pytest.mark.parametrize("batch", [1, 256, 257])
def test_counts_of_many_elements(ccc, oracle, batch):
    """Counters of every batch element, up to and past what a pinned block holds (256)."""
    t0, t1, m = cases.random_soup(24, seed=4, motion=0.2)
    rb, rt, _, _ = oracle.bvh(t0, t1)
    _, _, cnt, _, _, counts = oracle.compute_impulses(rb, rt, t0, t1, m)
    one = [_t(np.ascontiguousarray(np.broadcast_to(a, (batch, *a.shape)))) for a in (rb, rt, t0, t1, m)]
    out = ccc.compute_impulses(*one, 24, 16)
    assert ccc.last_counts() == [[counts[k] for k in ("candidates", "subprims", "roots", "collisions")]] * batch
    np.testing.assert_array_equal(_np(out[2]), np.broadcast_to(cnt, (batch, *cnt.shape)))


def test_counts_from_several_threads(ccc, oracle):
    """Calls of four threads on their own streams, each reading its own counters."""
    import threading

    import torch
    args, want, bad = [], [], []
    for k in range(4):
        t0, t1, m = cases.random_soup(40 + 30 * k, seed=k, motion=0.2)
        rb, rt, _, _ = oracle.bvh(t0, t1)
        counts = oracle.compute_impulses(rb, rt, t0, t1, m)[5]
        args.append([_t(a[None]) for a in (rb, rt, t0, t1, m)])
        want.append([[counts[c] for c in ("candidates", "subprims", "roots", "collisions")]])
    torch.cuda.synchronize()

    def work(k):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(30):
                ccc.compute_impulses(*args[k], 200, 16)
                if ccc.last_counts() != want[k]:
                    bad.append(k)

    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


@pytest.mark.parametrize("n", [2, 65, 300])
def test_index_tree_in_a_fitted_context(ccc, oracle, n):
    """A context that fits its trees walks every tree: the index tree's pairs are the same."""
    t0, t1, _ = cases.random_soup(n, seed=n + 9)
    rb, rt, _, _ = oracle.bvh(t0, t1)
    pairs, total = oracle.traverse(rb, rt, 0.0)
    ccc.set_morton_mode(1)
    try:
        rows, k = _mincol(ccc, rb, rt, t0, t1, total // n + 2)
    finally:
        ccc.set_morton_mode(0)
    assert k == total
    np.testing.assert_array_equal(rows, sorted_rows(oracle.mincol(t0, t1, pairs)))
