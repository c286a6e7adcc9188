"""The narrow phase's cubic solver inside, at and outside the coefficient range in which it
shares its reciprocals: the oracle's roots, bit for bit."""
import numpy as np
import pytest

from tests.test_gpu_device_math import _oracle_kept, _same_bits, dmath  # noqa: F401

pytestmark = pytest.mark.gpu


def _rooted(rng, n):
    """Cubics with a root in [0, 1] at most, scaled over the range and past its ends."""
    out = []
    for _ in range(n):
        s = 2.0 ** rng.uniform(-50, 44) * rng.choice([-1, 1])
        if rng.random() < 0.5:
            out.append(np.poly(rng.uniform(-0.5, 1.5, 3) * 10.0 ** rng.integers(-3, 2)) * s)
        else:
            p, q = rng.uniform(0, 1), rng.uniform(0.01, 10)
            out.append(np.polymul([1.0, -p], [1.0, rng.uniform(-1, 1), q]) * s)
    return out


def _edges(rng, n):
    """Coefficients over all magnitudes around the range's limits, zeros among them."""
    lim = np.array([2.0**20, 2.0**40, 2.0**-60, 2.0**-100, 1e-16, 1.0])
    out = []
    for _ in range(n):
        c = 2.0 ** rng.uniform(-115, 50, 4) * rng.choice([-1, 1], 4)
        c[0] = 2.0 ** rng.uniform(-53.2, 24) * rng.choice([-1, 1])
        for k in range(4):
            if rng.random() < 0.2:
                c[k] = np.nextafter(rng.choice(lim), rng.choice([0, 1e300])) * rng.choice([-1, 1])
            elif rng.random() < 0.1:
                c[k] = rng.choice([0.0, -0.0, 5e-324, 1e-310])
        out.append(c)
    return out


@pytest.mark.parametrize("make,n", [(_rooted, 20000), (_edges, 20000)])
def test_cubic_roots_over_the_shared_range(dmath, oracle, make, n):  # noqa: F811
    _, _, run = dmath
    coef = np.array(make(np.random.default_rng(21), n), np.float64)
    got = run(5, coef, per=4).reshape(-1, 4)
    kept = 0
    for c, g in zip(coef, got):
        want = _oracle_kept(oracle, c)
        assert int(g[0]) == len(want), (c, g, want)
        assert _same_bits(g[1:1 + len(want)], want), (c, g, want)
        kept += len(want)
    assert kept > n // 100
