"""fg_sort_pairs_ws around 786,432 keys, above which a tile's keys are ranked by
512 lanes in place of 1,024, against numpy's stable sort, exactly."""
import numpy as np
import pytest

from test_gpu_sort_shapes import _sorted

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [786431, 786432, 786433, 788481, 1200001])
@pytest.mark.parametrize("bits", [7, 16, 25])
def test_sizes_match_stable_sort(fglib, n, bits):
    rng = np.random.default_rng(n + bits)
    key = np.repeat(rng.integers(0, 1 << bits, n // 3 + 1), 3)[:n].astype(np.uint32)
    key[::5] = rng.integers(0, 1 << bits, len(key[::5]))
    order = np.argsort(key, kind="stable").astype(np.uint32)
    k, v = _sorted(fglib, key, bits)
    assert np.array_equal(v, order)
    assert np.array_equal(k, key[order])
