"""fg_body_reduce_f64 of bodies of all sizes around its levels (none, one, a
wavefront, a workgroup of 1,024 lanes and more): the pairwise FP64 sums over
1,024 lanes, level by level, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = (1, 0, 2, 8, 63, 64, 65, 127, 128, 129, 512, 513, 1023, 1024, 1025, 3000, 0, 20001)


def _sum(v):
    a = np.zeros((1024, 3))
    for i in range(0, len(v), 1024):
        part = v[i:i + 1024, :3].astype(np.float64)
        a[:len(part)] += part
    while len(a) > 1:
        a = a[:len(a) // 2] + a[len(a) // 2:]
    return a[0]


def test_sums_of_all_sizes(fglib):
    L = fglib.load()
    rng = np.random.default_rng(3)
    offsets = np.concatenate([[0], np.cumsum(SIZES)]).astype(np.uint32)
    f, t = (np.float32(10.0) ** rng.integers(-6, 6, (offsets[-1], 4)) * rng.normal(size=(offsets[-1], 4)) for _ in range(2))
    f, t = f.astype(np.float32), t.astype(np.float32)
    d = [fglib.DeviceArray.from_numpy(a) for a in (f, t, offsets)]
    out = [fglib.DeviceArray((len(SIZES), 4), np.float64) for _ in range(2)]
    acc = [fglib.DeviceArray((len(SIZES), 4), np.float32) for _ in range(2)]
    fglib.check(L.fg_body_reduce_f64(d[0].ptr, d[1].ptr, d[2].ptr, len(SIZES), out[0].ptr, out[1].ptr, acc[0].ptr,
                                     acc[1].ptr), "sums")
    for v, o, a in zip((f, t), out, acc):
        want = np.stack([_sum(v[lo:hi]) for lo, hi in zip(offsets[:-1], offsets[1:])])
        assert np.array_equal(o.numpy()[:, :3], want)
        assert np.array_equal(a.numpy()[:, :3], want.astype(np.float32))
