"""The boxes by which the candidate search groups queries: each group of 16 consecutive leaves is
split where that makes its two boxes smallest, whatever the other groups of its wave do."""
import ctypes

import numpy as np
import pytest

from tests import cases
from tests.test_gpu_parity import _np, _t
from tests.test_host import LIB

pytestmark = pytest.mark.gpu
Q = 16


def _groups(ccc, boxes, check=None):
    """chunks and groups of the leaf boxes [n, 6] as the library makes them."""
    import torch
    lib = ctypes.CDLL(LIB)
    P = ctypes.c_void_p
    lib.ccc_context_create.argtypes = [ctypes.POINTER(P), ctypes.c_int, P, P, P]
    lib.ccc_debug_query_groups.argtypes = [P, P, P, ctypes.c_int64, ctypes.c_int32, P, P, P]
    lib.ccc_context_destroy.argtypes = [P]
    ctx = P()
    assert lib.ccc_context_create(ctypes.byref(ctx), torch.cuda.current_device(), None, None, None) == 0
    n = len(boxes)
    nc = -(-n // 64)
    bb = _t(np.concatenate([np.full((n - 1, 6), np.nan, boxes.dtype), boxes]))
    chunks, groups = bb.new_zeros((nc, 6)), bb.new_zeros((4 * nc, 2, 6))
    torch.cuda.synchronize()
    byte = None if check is None else _t(check.astype(np.uint8))
    st = lib.ccc_debug_query_groups(ctx, bb.data_ptr(), None if byte is None else byte.data_ptr(), n, 1 if bb.dtype == torch.float64 else 0,
                                    chunks.data_ptr(), groups.data_ptr(), None)
    assert st == 0
    torch.cuda.synchronize()
    lib.ccc_context_destroy(ctx)
    return _np(chunks), _np(groups)


def _union(b):
    return np.concatenate([np.fmin.reduce(b[:, :3], 0), np.fmax.reduce(b[:, 3:], 0)])


def _extent(b):
    d = (b[3:] - b[:3]).astype(np.float32)
    return max(d[0] + d[1] + d[2], np.float32(0))


def _split(b):
    """Where the 16 boxes are split (15: not at all), in the library's single-precision terms."""
    cost = np.array([_extent(_union(b[:k + 1])) + _extent(_union(b[k + 1:])) for k in range(Q - 1)], np.float32)
    at = int(cost.argmin())
    return at if cost[at] < np.float32(0.75) * _extent(_union(b)) else Q - 1


def _boxes(kind, n, dtype):
    if kind == "cloth":
        t0, t1, _ = cases.folded(n, seed=3)
        p = np.concatenate([t0, t1], 1)
        return np.concatenate([p.min(1), p.max(1)], 1).astype(dtype)
    rng = np.random.default_rng(n)
    # strips of random lengths, each somewhere else: most groups span two or three
    strip = np.cumsum(rng.random(n) < 0.11)
    c = rng.random((strip.max() + 1, 3))[strip] + 0.01 * rng.random((n, 3))
    return np.concatenate([c, c + 0.01 * rng.random((n, 3))], 1).astype(dtype)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind, n", [("cloth", 16), ("cloth", 23), ("strips", 1), ("strips", 15), ("strips", 17), ("strips", 64),
                                     ("strips", 200), ("strips", 4099)])
def test_each_group_has_its_own_split(ccc, kind, n, dtype):
    boxes = _boxes(kind, n, dtype)
    n = len(boxes)
    chunks, groups = _groups(ccc, boxes)
    padded = np.concatenate([boxes, np.repeat(boxes[-1:], -n % 64, 0)])
    split = 0
    for c in range(len(chunks)):
        np.testing.assert_array_equal(chunks[c], _union(padded[64 * c:64 * c + 64]))
    for g in range(len(groups)):
        b = padded[Q * g:Q * g + Q]
        at = _split(b)
        split += at < Q - 1
        want = (_union(b[:at + 1]), _union(b[at + 1:])) if at < Q - 1 else (_union(b), _union(b))
        np.testing.assert_array_equal(groups[g], np.stack(want), err_msg=f"group {g}")
    assert split > 0 or n < 64


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n, share", [(1, 0.0), (40, 0.0), (40, 0.1), (64, 0.5), (1000, 0.02), (1000, 0.2), (1000, 1.0), (4099, 0.01)])
def test_groups_of_checked_leaves_only(ccc, n, share, dtype):
    """A partial query's groups cover its checked triangles and no others."""
    boxes = _boxes("strips", n, dtype)
    check = np.random.default_rng(n + 1).random(n) < share
    chunks, groups = _groups(ccc, boxes, check)
    at = np.minimum(np.arange(len(groups) * Q), n - 1)
    padded, on = boxes[at].copy(), check[at]
    for c in range(len(chunks)):
        np.testing.assert_array_equal(chunks[c], _union(padded[64 * c:64 * c + 64]))
    padded[~on] = [np.inf] * 3 + [-np.inf] * 3
    with np.errstate(invalid="ignore"):
        for g in range(len(groups)):
            b = padded[Q * g:Q * g + Q]
            k = _split(b)
            want = (_union(b[:k + 1]), _union(b[k + 1:])) if k < Q - 1 else (_union(b), _union(b))
            np.testing.assert_array_equal(groups[g], np.stack(want), err_msg=f"group {g}")
