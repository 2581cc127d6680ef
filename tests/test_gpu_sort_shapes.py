"""fg_sort_pairs_ws around the sizes where its tiles and launches change: a
wavefront, a tile of 2,048 keys, 64 tiles (above them the counts are scanned),
1,572,864 keys (above them tiles of 4,096), each against numpy's stable sort,
exactly."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _sorted(fglib, key, bits):
    L, n = fglib.load(), len(key)
    size = L.fg_sort_workspace_size(n, bits)
    dk, dv, ws = fglib.DeviceArray.from_numpy(key), fglib.DeviceArray((n,), np.uint32), fglib.DeviceArray((size,), np.uint8)
    fglib.check(L.fg_sort_pairs_ws(dk.ptr, dv.ptr, n, bits, ws.ptr, size, 1), "fg_sort_pairs_ws")
    return dk.numpy(), dv.numpy()


@pytest.mark.parametrize("n", [1, 63, 65, 2047, 2048, 2049, 131071, 131072, 131073, 133121, 1572864, 1572865, 1579009])
@pytest.mark.parametrize("kind,bits", [("random", 6), ("random", 22), ("runs", 16), ("falling", 21), ("equal", 13)])
def test_sizes_match_stable_sort(fglib, n, kind, bits):
    rng = np.random.default_rng(n + bits)
    key = {"random": lambda: rng.integers(0, 1 << bits, n),
           "runs": lambda: np.repeat(rng.integers(0, 1 << bits, n // 8 + 1), 8)[:n],
           "falling": lambda: (1 << bits) - 1 - (np.arange(n) % (1 << bits)),
           "equal": lambda: np.full(n, (1 << bits) - 1)}[kind]().astype(np.uint32)
    order = np.argsort(key, kind="stable").astype(np.uint32)
    k, v = _sorted(fglib, key, bits)
    assert np.array_equal(v, order)
    assert np.array_equal(k, key[order])


def test_workspace_of_more_keys_serves_fewer(fglib):
    """The workspace size does not fall where the tiles grow."""
    L = fglib.load()
    for bits in (8, 16, 22, 32):
        sizes = [L.fg_sort_workspace_size(n, bits) for n in (1, 2048, 131073, 1572863, 1572864, 1572865, 1580000, 4194304,
                                                             4194305, 8388608)]
        assert sizes == sorted(sizes)
