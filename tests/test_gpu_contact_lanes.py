"""Body forces from the fluid where the walk over groups of lanes can go
wrong: buckets longer than one pass of eight and than the list of spheres
within reach, stencils of one cell and of more than one batch of 32, partial
wavefronts, and tables whose size is no power of two.  Same IEEE operations
in the same order as the oracle, contraction off: <= 1 ulp, as for the other
body forces."""
import numpy as np
import pytest

from fluidgrid_amd import abi, scenes
from test_gpu_rigid import _dev, _ulp_diff

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,buckets,relation,reach", [
    (1, 4096, (1, 1, 1), 0.02),
    (9, 1000, (1, 1, 1), 0.02),
    (67, 5, (1, 1, 1), 0.02),
    (200, 64, (1, 1, 1), 0.08),
    (31, 3, (0, 0, 0), 0.08),
    (41, 1000, (2, 1, 2), 0.04),
    (8, 1, (3, 2, 0), 0.08),
])
def test_long_cells_and_wide_stencils_match_oracle(fglib, orc, m, buckets, relation, reach):
    L = fglib.load()
    s = scenes.dam_break((8, 8, 8), 0.02, (1.0, 1.0, 1.0), 1e-4)
    fglib.init_params(s.common, s.kernels, abi.KEY_REF_XOR)
    rng = np.random.default_rng(m + buckets)
    n, cell = 700, 0.021
    pos = np.zeros((n, 4), np.float32)
    vel = np.zeros((n, 4), np.float32)
    pos[:, :3], pos[:, 3] = rng.uniform(0.0, 0.1, (n, 3)), 1.0
    vel[:, :3] = rng.normal(0.0, 0.2, (n, 3))
    key, pid = orc.hash_keys(pos, buckets, (cell,) * 3, s.common, abi.KEY_REF_XOR)
    start, end, spos, svel = orc.cell_offsets(*orc.sort_pairs(key, pid), pos, vel, buckets)
    world = np.zeros((m, 4), np.float32)
    world[:, :3] = rng.uniform(0.0, 0.1, (m, 3))
    bvel = np.array([[0.05, -0.3, 0.02, 0.0]], np.float32)
    cm = np.array([[0.05, 0.05, 0.05, 0.0]], np.float32)
    d = {k: _dev(fglib, v) for k, v in dict(w=world, bv=bvel, cm=cm, spos=spos, svel=svel, start=start,
                                           end=end).items()}
    f, t = fglib.DeviceArray((m, 4), np.float32), fglib.DeviceArray((m, 4), np.float32)
    fglib.check(L.fg_body_forces_from_fluid(d["w"].ptr, d["bv"].ptr, d["cm"].ptr, f.ptr, t.ptr, m, 1, reach,
                                            d["spos"].ptr, d["svel"].ptr, d["start"].ptr, d["end"].ptr, n, 0.002,
                                            abi.Float3(cell, cell, cell), buckets, abi.Int3(*relation), -2000.0,
                                            -50.0), "forces from fluid")
    of, ot = orc.body_forces_from_fluid(world, bvel, cm, reach, spos, svel, start, end, 0.002,
                                        orc.grid_of_bodies(cell, buckets), relation, -2000.0, -50.0)
    assert np.count_nonzero(of[:, 0])
    assert _ulp_diff(f.numpy(), of).max() <= 1
    assert _ulp_diff(t.numpy(), ot).max() <= 1
