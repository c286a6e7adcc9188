"""Calls through torch's allocator when device memory is short: what a call can do without it
does without, and what it cannot raises torch's own error and leaves the next call whole."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
MIB = 1 << 20


class limited:
    """At most `more` bytes beyond what torch holds now, for the time of the block."""

    def __init__(self, more):
        self.more = more

    def __enter__(self):
        import torch
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        total = torch.cuda.get_device_properties(0).total_memory
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + self.more) / total)

    def __exit__(self, *exc):
        import torch
        torch.cuda.set_per_process_memory_fraction(1.0)
        torch.cuda.empty_cache()


def _rows(n, dtype):
    import torch
    g = torch.Generator(device="cuda").manual_seed(5)

    def rand(*shape):
        return torch.rand(shape, generator=g, dtype=torch.float64, device="cuda")

    x = torch.randint(0, n - 1, (n,), generator=g, device="cuda").sort().values
    rows = torch.stack([x, x + 1, torch.randint(0, 15, (n,), generator=g, device="cuda")], 1)[None].contiguous()
    t0 = rand(1, n, 3, 3)
    return rows, rand(1, n, 1).to(dtype), t0.to(dtype), (t0 + 0.1 * rand(1, n, 3, 3)).to(dtype), (0.5 + rand(1, n, 3)).to(dtype)


@pytest.mark.parametrize("dtype, room", [("float64", 52), ("float32", 36)])
def test_given_rows_without_room_for_lines(ccc, dtype, room):
    """Lines for 200k triangles take a segment of 38 MiB, the outputs 28 to 48 in double and at
    most 20 in float: with 52 or 36 MiB the sums go straight to the outputs.  Sums of k shares in
    another order differ by at most 2 k ulp of their sizes' sum."""
    import torch
    args = _rows(200_000, getattr(torch, dtype))
    want = [a.cpu() for a in ccc.compute_impulses_from_collisions(*args)]
    with limited(room * MIB):
        got = [a.cpu() for a in ccc.compute_impulses_from_collisions(*args)]
    assert torch.equal(got[2], want[2])
    k = int(want[2].max())
    for a, b in zip(got[:2], want[:2]):
        fin = torch.isfinite(b)
        assert torch.equal(torch.isfinite(a), fin)
        assert float((a - b)[fin].abs().max()) <= 2 * k * k * np.finfo(dtype).eps * float(b[fin].abs().max())


def test_no_room_for_a_workspace(ccc):
    import torch
    _, _, t0, t1, m = _rows(200_000, torch.float64)
    t0, t1 = 100 * t0[:, :, :1] + 0.1 * t0, 100 * t0[:, :, :1] + 0.1 * t1
    bb, tree = ccc.bvh_motion(t0, t1)
    want = ccc.compute_impulses(bb, tree, t0, t1, m, 4, 4)[2].cpu()
    with limited(52 * MIB):
        with pytest.raises(torch.OutOfMemoryError):
            ccc.compute_impulses(bb, tree, t0, t1, m, 4, 4)
    assert torch.equal(ccc.compute_impulses(bb, tree, t0, t1, m, 4, 4)[2].cpu(), want)
