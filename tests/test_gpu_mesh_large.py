"""Lattices beyond what one dimension of a launch holds (two points of a row a
lane): sampled points, the last ones and those around the launch's rows among
them, against the 64-bit oracle, and nothing is left unwritten.  Tolerance:
2e-5 for points farther than 1e-3 from every face's plane, as in
test_gpu_mesh.py (each term is an FP32 arc tangent of FP32 differences)."""
import numpy as np
import pytest

from fluidgrid_amd import abi
from oracle import mesh as om

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(813, 813, 813), (1, (1 << 14) + 1, 1 << 14)], ids=["cube", "one_a_row"])
def test_large_lattice(fglib, dims):
    L = fglib.load()
    v = np.array([[0.1, 0.1, 0.1], [0.9, 0.15, 0.2], [0.3, 0.85, 0.1], [0.35, 0.3, 0.9]], np.float32)
    t = np.array([[0, 2, 1], [0, 1, 3], [1, 2, 3], [2, 0, 3]], np.uint32)
    n, spacing = dims[0] * dims[1] * dims[2], np.float32(1.0 / max(dims))
    dv, dt = fglib.DeviceArray.from_numpy(v), fglib.DeviceArray.from_numpy(t)
    x0 = np.float32(0.35 if dims[0] == 1 else 0.0)
    out = fglib.DeviceArray((n,), np.float32)
    out.fill_u32(0xFFFFFFFF)  # NaN
    fglib.check(L.fg_mesh_winding_lattice(dv.ptr, len(v), dt.ptr, len(t), abi.f3(x0, 0.0, 0.0), float(spacing), *dims,
                                          out.ptr), "winding")
    fglib.check(None, "winding")
    w = out.numpy()
    out.free()
    assert not np.isnan(w).any()
    rng = np.random.default_rng(1)
    edge = (1 << 21) * 64 * (1 if dims[0] == 1 else 2)  # points of a full row of workgroups, about
    at = np.unique(np.concatenate([np.arange(64), n - 1 - np.arange(64), edge + np.arange(-300, 300),
                                   rng.integers(0, n, 2000)]))
    i = np.stack([at % dims[0], at // dims[0] % dims[1], at // (dims[0] * dims[1])], 1).astype(np.float32)
    pts = (i * spacing + np.array([x0, 0.0, 0.0], np.float32)).astype(np.float32)
    far = np.ones(len(at), bool)
    for a, b, c in v[t].astype(np.float64):
        normal = np.cross(b - a, c - a)
        far &= np.abs((pts - a) @ normal) > 1e-3 * np.linalg.norm(normal)
    want = om.winding(pts, v, t)
    assert far.sum() > 2000 and 0.02 < (want[far] > 0.5).mean() < 0.98
    assert np.max(np.abs(w[at] - want)[far]) <= 2e-5
