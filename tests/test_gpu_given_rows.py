"""compute_impulses_from_collisions where the split of its rows over waves changes."""
import numpy as np
import pytest

from tests import test_gpu_pairs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("m", [32, 63, 65, 16383, 16384, 16385])
def test_rows_at_the_edges_of_waves(ccc, oracle, m, dtype):
    """Two meshes' rows: 32 per wave up to 32,768 in all, 64 from there on."""
    test_gpu_pairs.test_impulses_of_given_rows(ccc, oracle, m, dtype)
