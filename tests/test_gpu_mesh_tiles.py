"""fg_mesh_winding_lattice where its split can go wrong: rows of one, of an odd
and of more points than a wavefront's, triangle counts around a tile's 1,024,
and triangles left out within and at the end of tiles.  Tolerance of the other
winding numbers: 2e-5 + 1e-8 a triangle, away from the triangles."""
import numpy as np
import pytest

from fluidgrid_amd import abi
from oracle import mesh as om

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(1, 1, 1), (2, 3, 5), (3, 1, 43), (131, 2, 1), (1, 70, 3)])
@pytest.mark.parametrize("ntris", [1, 1023, 1024, 1025, 2111])
def test_tiles_and_rows_match_oracle(fglib, dims, ntris):
    L = fglib.load()
    rng = np.random.default_rng(ntris + dims[0])
    # triangles of every size in the unit box; the lattice lies beside it and ends next to it
    centre = rng.uniform(0.0, 1.0, (ntris, 1, 3))
    size = 10.0 ** rng.uniform(-3.0, -0.3, (ntris, 1, 1))
    v = np.clip(centre + size * rng.normal(0.0, 1.0, (ntris, 3, 3)), 0.0, 1.0).astype(np.float32).reshape(-1, 3)
    t = np.arange(3 * ntris, dtype=np.uint32).reshape(-1, 3)
    bad = rng.random(ntris) < 0.05
    bad[-1] = ntris > 1
    t_bad = t.copy()
    t_bad[bad, rng.integers(0, 3, ntris)[bad]] = len(v) + rng.integers(0, 2, ntris)[bad]
    s = 0.01
    origin = np.array([0.3, 0.2, -0.02 - s * dims[2]], np.float32)
    dv, dt = fglib.DeviceArray.from_numpy(v), fglib.DeviceArray.from_numpy(t_bad)
    w = fglib.DeviceArray((dims[0] * dims[1] * dims[2],), np.float32)
    fglib.check(L.fg_mesh_winding_lattice(dv.ptr, len(v), dt.ptr, ntris, abi.Float3(*origin), s, *dims, w.ptr),
                "fg_mesh_winding_lattice")
    w64 = om.winding(om.lattice_points(origin, s, dims), v, t[~bad])
    assert np.abs(w.numpy() - w64).max() <= 2e-5 + 1e-8 * ntris
