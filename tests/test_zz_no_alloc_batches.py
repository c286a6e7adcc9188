"""Batches of many tiny meshes: what they take of the allocation-free entry point's scratch
array and of device memory follows their pairs."""
import numpy as np
import pytest

from tests import cases
from tests.test_gpu_parity import _np, _renumbered_internal_tree, _t
from tests.test_zz_no_alloc import CCC_ERR_NO_MEMORY, _call, capi  # noqa: F401

pytestmark = pytest.mark.gpu


def _batch(oracle, n, batch, foreign):
    t0, t1, m = cases.random_soup(n, seed=n, motion=0.3)
    bb, tree, _, _ = oracle.bvh(t0, t1)
    want = oracle.compute_impulses(bb, tree, t0, t1, m)
    if foreign:
        bb, tree = _renumbered_internal_tree(bb, tree, 2)
    one = [_t(a)[None].expand(batch, *a.shape).contiguous() for a in (bb, tree, t0, t1, m)]
    return one, want


# the largest batches: about 210 of the array's 256 MiB with the tree walk's 5 to 6 KiB per mesh
@pytest.mark.parametrize("n, batch, foreign", [(2, 2000, False), (2, 2300, False), (2, 30000, False), (5, 2300, True),
                                               (5, 30000, True), (24, 4000, False), (24, 4000, True)])
def test_noalloc_on_many_elements(ccc, oracle, capi, n, batch, foreign):  # noqa: F811
    args, want = _batch(oracle, n, batch, foreign)
    st, dv, dx, cnt, counts, err = _call(capi, capi[3], *args, n)
    assert st == 0, err
    w = tuple(want[5][k] for k in ("candidates", "subprims", "roots", "collisions"))
    assert set(counts) == {w}
    cnt = _np(cnt)
    np.testing.assert_array_equal(cnt, np.broadcast_to(want[2], cnt.shape))
    # one mesh's sums, whose terms come in any order: within 1e-9 as everywhere
    for got, ref in ((dv, want[0]), (dx, want[1])):
        fin = np.isfinite(ref)
        d = np.abs(_np(got)[:, fin] - ref[fin])
        assert d.size == 0 or d.max() <= 1e-9 * max(np.abs(ref[fin]).max(), 1e-300)


@pytest.mark.parametrize("batch", [1, 63, 64, 65, 20000])
def test_device_memory_of_many_elements(ccc, oracle, batch):
    """At most 12 KiB per mesh of two triangles beyond the call's outputs (its list holds one
    batch of 64 pairs, 3.9 KiB), and 64 KiB for a call's small buffers."""
    import torch
    args, want = _batch(oracle, 2, batch, False)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    held = torch.cuda.memory_allocated()
    dv, dx, cnt = ccc.compute_impulses(*args, 2, 16)
    outputs = sum(a.numel() * a.element_size() for a in (dv, dx, cnt))
    assert torch.cuda.max_memory_allocated() - held - outputs <= batch * 12 * 1024 + 65536
    cnt = _np(cnt)
    np.testing.assert_array_equal(cnt, np.broadcast_to(want[2], cnt.shape))


def test_noalloc_with_a_list_in_pieces(ccc, oracle, capi):  # noqa: F811
    """A candidate capacity that leaves the scratch array room for a few batches of pairs only:
    the same result, by the index tree and by the walk, whose buffers then make the room."""
    t0, t1, m = cases.random_soup(120, seed=1, motion=0.3)
    bb, tree, _, _ = oracle.bvh(t0, t1)
    want = oracle.compute_impulses(bb, tree, t0, t1, m)
    k = tuple(want[5][c] for c in ("candidates", "subprims", "roots", "collisions"))
    total = 256 << 20
    for foreign in (False, True):
        fb, ft = _renumbered_internal_tree(bb, tree, 2) if foreign else (bb, tree)
        args = [_t(a[None]) for a in (fb, ft, t0, t1, m)]
        seen = set()
        for left in (6 << 10, 32 << 10, 64 << 10, 96 << 10, 256 << 10):
            st, dv, dx, cnt, counts, err = _call(capi, capi[3], *args, (total - left) // (8 * 120))
            seen.add(st & 0xff)
            if st & 0xff:
                assert st & 0xff == CCC_ERR_NO_MEMORY and b"scratch" in err
                continue
            assert counts == [k]
            np.testing.assert_array_equal(_np(cnt)[0], want[2])
        assert seen == {0, CCC_ERR_NO_MEMORY}


def test_noalloc_with_the_deep_stack(ccc, oracle, capi):  # noqa: F811
    """A tree whose rows are numbered at random needs the walk's deep stack: in the scratch array
    its buffers and the list are then laid out again."""
    n = 40000
    rng = np.random.default_rng(31)
    c = rng.random((n, 3))
    key = np.zeros(n, np.int64)
    for bit in range(10):
        for a in range(3):
            key |= ((c[:, a] * 1024).astype(np.int64) >> bit & 1) << (3 * bit + a)
    c = c[np.argsort(key)][:, None]
    t0 = c + 0.01 * rng.standard_normal((n, 3, 3))
    t1 = t0 + 0.01 * rng.standard_normal((n, 3, 3))
    m = rng.uniform(0.5, 2.0, (n, 3))
    bb, tree, _, _ = oracle.bvh(t0, t1)
    args = [_t(a[None]) for a in (t0, t1, m)]
    ref = _call(capi, capi[2], _t(bb[None]), _t(tree[None]), *args, 64)
    bb, tree = (_t(a[None]) for a in _renumbered_internal_tree(bb, tree, 4))
    for fn in (capi[2], capi[3]):
        got = _call(capi, fn, bb, tree, *args, 64)
        assert got[0] & 0xff == 0, got[5]
        assert got[4] == ref[4] and ref[4][0][3] > 0
        np.testing.assert_array_equal(_np(got[3]), _np(ref[3]))
