"""Body forces from the fluid around the stencil sizes where the walk passes
from a sphere a lane to a cell a lane: 45 and 63 cells on positional keys, 125
and 147 on hashed ones.  Same IEEE operations in the same order as the oracle,
contraction off: <= 1 ulp, as for the other body forces."""
import numpy as np
import pytest

from fluidgrid_amd import abi, scenes
from test_gpu_rigid import _dev, _ulp_diff

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [abi.KEY_LINEAR, abi.KEY_REF_XOR])
@pytest.mark.parametrize("m,buckets,relation,reach", [
    (67, 4096, (2, 1, 1), 0.03),
    (67, 4096, (1, 3, 1), 0.03),
    (1, 4096, (2, 2, 2), 0.02),
    (131, 1000, (2, 2, 2), 0.04),
    (9, 7, (3, 1, 3), 0.08),
    (33, 4096, (3, 3, 3), 0.02),
])
def test_wide_stencils_match_oracle(fglib, orc, mode, m, buckets, relation, reach):
    L = fglib.load()
    s = scenes.dam_break((8, 8, 8), 0.02, (1.0, 1.0, 1.0), 1e-4)
    fglib.init_params(s.common, s.kernels, mode)
    rng = np.random.default_rng(m + buckets)
    lo = np.array([*s.common.volume_min], np.float32)  # stencils of the corner's cells leave the grid
    cell, n = (s.common.cell_size if mode == abi.KEY_LINEAR else abi.Float3(0.021, 0.021, 0.021)), 700
    if mode == abi.KEY_LINEAR:
        buckets, grid = s.common.num_buckets(), orc.grid_of_fluid(s.common, mode)
    else:
        grid = orc.grid_of_bodies(0.021, buckets)
    pos = np.zeros((n, 4), np.float32)
    vel = np.zeros((n, 4), np.float32)
    pos[:, :3], pos[:, 3] = lo + rng.uniform(0.0, 0.1, (n, 3)), 1.0
    vel[:, :3] = rng.normal(0.0, 0.2, (n, 3))
    key, pid = orc.hash_keys(pos, buckets, tuple(cell), s.common, mode)
    start, end, spos, svel = orc.cell_offsets(*orc.sort_pairs(key, pid), pos, vel, buckets)
    world = np.zeros((m, 4), np.float32)
    world[:, :3] = lo + rng.uniform(0.0, 0.1, (m, 3))
    bvel = np.array([[0.05, -0.3, 0.02, 0.0]], np.float32)
    cm = np.append(lo + np.float32(0.05), np.float32(0.0))[None].astype(np.float32)
    d = {k: _dev(fglib, v) for k, v in dict(w=world, bv=bvel, cm=cm, spos=spos, svel=svel, start=start,
                                           end=end).items()}
    f, t = fglib.DeviceArray((m, 4), np.float32), fglib.DeviceArray((m, 4), np.float32)
    fglib.check(L.fg_body_forces_from_fluid(d["w"].ptr, d["bv"].ptr, d["cm"].ptr, f.ptr, t.ptr, m, 1, reach,
                                            d["spos"].ptr, d["svel"].ptr, d["start"].ptr, d["end"].ptr, n, 0.002,
                                            cell, buckets, abi.Int3(*relation), -2000.0,
                                            -50.0), "forces from fluid")
    of, ot = orc.body_forces_from_fluid(world, bvel, cm, reach, spos, svel, start, end, 0.002,
                                        grid, relation, -2000.0, -50.0)
    assert np.count_nonzero(of[:, 0])
    assert _ulp_diff(f.numpy(), of).max() <= 1
    assert _ulp_diff(t.numpy(), ot).max() <= 1
