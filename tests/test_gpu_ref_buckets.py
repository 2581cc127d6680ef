"""The reference-arithmetic kernels over buckets of 0 to 70 particles, around
the 16 up to which the eight-lane force kernel walks four buckets of a lane as
one list and the 32 of one mask, against the FP32 oracle (tolerances of
test_gpu_sph.py)."""
import numpy as np
import pytest

from fluidgrid_amd import abi
from test_gpu_ref_lanes import _scene
from test_gpu_sph import check_density, check_velocity, gpu_density, gpu_forces, grid_cpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("key_mode", [abi.KEY_REF_XOR, abi.KEY_LINEAR])
@pytest.mark.parametrize("sizes", [(15, 16), (16, 17), (0, 1, 16, 31), (32, 33, 3), (70, 5)])
def test_bucket_lengths_match_oracle(fglib, orc, key_mode, sizes):
    s = _scene(1, key_mode)
    rng = np.random.default_rng(sum(sizes))
    cell = s.common.cell_size.x
    corner = s.pos[0, :3] + 8.0 * cell
    corner = np.floor(corner / cell) * cell
    pos = []
    for c in range(64):  # a block of 4 x 4 x 4 cells
        base = corner + cell * np.array([c % 4, (c // 4) % 4, c // 16])
        pos.append(base + cell * rng.uniform(0.05, 0.95, (sizes[c % len(sizes)], 3)))
    p = np.concatenate(pos)
    n = len(p)
    s.pos = np.ones((n, 4), np.float32)
    s.pos[:, :3] = p
    s.vel = np.zeros((n, 4), np.float32)
    s.vel[:, :3] = rng.normal(0.0, 1.0, (n, 3))
    s.fluid.max_particles = n
    sk, sp, start, end, spos, svel = grid_cpu(orc, s)
    rp = gpu_density(fglib, s, spos, start, end, abi.MATH_REFERENCE)
    check_density(rp, orc.density(spos, start, end, s.fluid, s.common, s.kernels, s.key_mode), s)
    v_ref, acc, _ = orc.forces(spos, svel, rp, start, end, sp, s.fluid, s.common, s.kernels, s.key_mode,
                               v_out_init=s.vel, want_acc=True)
    _, _, mag = orc.forces(spos, svel, rp.astype(np.float64), start, end, sp, s.fluid, s.common, s.kernels,
                           s.key_mode, f64=True, want_mag=True)
    vel, _ = gpu_forces(fglib, s, spos, svel, rp, start, end, sp, abi.MATH_REFERENCE)
    check_velocity(vel, v_ref.astype(np.float64), acc, mag, sp, s.common.deltaTimeIntegration)
