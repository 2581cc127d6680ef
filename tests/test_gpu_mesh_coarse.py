"""Winding numbers of coarse meshes, where most pairs of a point and a triangle
are near: the mean error against the 64-bit oracle is no larger than that of
the plain FP32 formula (exact roots, every operation rounded, the arc tangent
correctly rounded) summed in 64 bits.  Meshes on both sides of the kernel's
rule for few triangles."""
import numpy as np
import pytest

from fluidgrid_amd import abi, mesh
from oracle import mesh as om

pytestmark = pytest.mark.gpu

F = np.float32
MESHES = {
    "box_12": lambda: mesh.box_mesh((-0.49, -0.49, -0.49), (0.49, 0.49, 0.49)),
    "sphere_20": lambda: mesh.icosphere_mesh(0.35, 0),
    "sphere_80": lambda: mesh.icosphere_mesh(0.35, 1),
    "torus_126": lambda: mesh.torus_mesh(0.3, 0.1, 9, 7),
    "torus_130": lambda: mesh.torus_mesh(0.3, 0.1, 13, 5),
    "sphere_320": lambda: mesh.icosphere_mesh(0.35, 2),
}


def _plain(p, v, t):
    def dot(x, y):
        return x[:, 0] * y[:, 0] + x[:, 1] * y[:, 1] + x[:, 2] * y[:, 2]

    acc = np.zeros(len(p))
    for tri in t:
        a, b, c = (v[k] - p for k in tri)
        la, lb, lc = (np.sqrt(dot(x, x)) for x in (a, b, c))
        det = (a[:, 0] * (b[:, 1] * c[:, 2] - b[:, 2] * c[:, 1]) + a[:, 1] * (b[:, 2] * c[:, 0] - b[:, 0] * c[:, 2]) +
               a[:, 2] * (b[:, 0] * c[:, 1] - b[:, 1] * c[:, 0]))
        den = la * lb * lc + dot(a, b) * lc + dot(b, c) * la + dot(c, a) * lb
        assert det.dtype == F and den.dtype == F
        acc += np.arctan2(det.astype(np.float64), den).astype(F)
    return (acc / (2.0 * np.pi)).astype(F)


@pytest.mark.parametrize("which", list(MESHES))
def test_mean_error(fglib, which):
    L = fglib.load()
    v, t = MESHES[which]()
    v, t = np.ascontiguousarray(v, F), np.ascontiguousarray(t, np.uint32)
    side = 41
    origin, spacing = np.array([-0.5, -0.4987, -0.4979], F), F(1.0 / side)
    dv, dt = fglib.DeviceArray.from_numpy(v), fglib.DeviceArray.from_numpy(t)
    out = fglib.DeviceArray((side ** 3,), F)
    fglib.check(L.fg_mesh_winding_lattice(dv.ptr, len(v), dt.ptr, len(t), abi.f3(*origin), float(spacing), side, side,
                                          side, out.ptr), "winding")
    p = om.lattice_points(origin, spacing, (side, side, side))
    exact = om.winding(p, v, t)

    def mean(w):
        e = np.abs(w.astype(np.float64) - exact)
        return e[e < 1e-3].mean()  # (a point on the surface may go either way)

    assert mean(out.numpy()) <= mean(_plain(p, v, t))
