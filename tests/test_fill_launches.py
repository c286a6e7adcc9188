"""The launches that clear a call's outputs: a launch holds fewer than 2^32 work items, 64 GiB at
16 bytes each, and outputs may be larger.  The arithmetic runs on the host; one test on the
card clears such an output through a query."""
import ctypes

import numpy as np
import pytest

from tests import cases
from tests.test_host import LIB

GIB = 1 << 30


@pytest.mark.parametrize("sizes", [[], [0], [4], [4096], [4100, 0, 12], [32 * GIB], [32 * GIB + 4], [64 * GIB - 4096], [64 * GIB],
                                   [64 * GIB + 4], [64, 256, 8192, 74 * GIB + 360], [40 * GIB, 40 * GIB, 40 * GIB], [250 * GIB]])
def test_launches_cover_every_block_once(sizes):
    fn = ctypes.CDLL(LIB).ccc_debug_fill_launches
    fn.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p, ctypes.c_int]
    b = np.array(sizes or [0], np.int64)
    out = np.zeros((64, 2), np.int64)
    k = fn(b.ctypes.data, len(sizes), out.ctypes.data, 64)
    assert 0 <= k <= 64
    at = 0
    for base, n in out[:k]:
        assert base == at and 0 < n * 256 < 1 << 32
        at += n
    assert at == sum(-(-s // 4096) for s in sizes)


@pytest.mark.gpu
def test_output_of_more_than_64_gib(ccc, oracle):
    """Rows of two triangles' sub-primitive pairs in an output of 69 GiB: the rows, then -1."""
    import torch
    if torch.cuda.mem_get_info()[0] < 100 * GIB:
        pytest.skip("needs 100 GiB of free device memory")
    t0, t1, _ = cases.random_soup(2, seed=3, motion=2.0)
    rb, rt, _, _ = oracle.bvh(t0, t1)
    pairs, total = oracle.traverse(rb, rt, 0.0)
    want = oracle.mincol(t0, t1, pairs)
    assert total == 1 and len(want) > 0
    cap = 103_000_000
    args = [torch.from_numpy(a[None]).cuda() for a in (rb, rt, t0, t1)]
    rows = ccc.find_mincol_cand(*args, cap)
    rows = rows[0] if isinstance(rows, (list, tuple)) else rows
    assert rows.numel() * 8 > 64 * GIB
    flat = rows.view(-1, 3)
    k = len(want)
    got = flat[:k].cpu().numpy()
    assert sorted(map(tuple, got.tolist())) == sorted(map(tuple, np.asarray(want).tolist()))
    for part in flat[k:].split(1 << 28):
        assert bool((part == -1).all())
    del rows, flat, part
    torch.cuda.empty_cache()
