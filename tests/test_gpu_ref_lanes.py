"""The reference-arithmetic density and force kernels at the sizes where the
lanes a particle takes change or a group is incomplete, against the FP32
oracle (tolerances of test_gpu_sph.py, stated there per quantity)."""
import numpy as np
import pytest

from fluidgrid_amd import abi, scenes
from test_gpu_sph import check_density, check_velocity, gpu_density, gpu_forces, grid_cpu

pytestmark = pytest.mark.gpu


def _scene(n, key_mode):
    """The reference application's block with n particles, thinned or
    continued to n, in motion; every seventh inactive where there are enough."""
    s = scenes.appmain_scene()
    spacing = s.info["spacing"]
    side = max(2, int(round(n ** (1 / 3))))
    i = np.arange(n)
    rng = np.random.default_rng(n)
    s.pos = np.ones((n, 4), np.float32)
    s.pos[:, :3] = np.stack([i % side, i // (side * side), (i // side) % side], 1) * spacing - 19.0
    s.pos[:, :3] += rng.uniform(-0.2 * spacing, 0.2 * spacing, (n, 3))
    s.vel = np.zeros((n, 4), np.float32)
    s.vel[:, :3] = rng.normal(0.0, 1.0, (n, 3))
    s.fluid.max_particles = n
    s.key_mode = key_mode
    return s


@pytest.mark.parametrize("key_mode", [abi.KEY_REF_XOR, abi.KEY_LINEAR])
@pytest.mark.parametrize("n", [1, 7, 9, 65, 3001, 163840, 163841])
def test_reference_kernels_match_oracle(fglib, orc, n, key_mode):
    s = _scene(n, key_mode)
    sk, sp, start, end, spos, svel = grid_cpu(orc, s)
    ref_rp = orc.density(spos, start, end, s.fluid, s.common, s.kernels, s.key_mode)
    rp = gpu_density(fglib, s, spos, start, end, abi.MATH_REFERENCE)
    check_density(rp, ref_rp, s)
    v_ref, acc, _ = orc.forces(spos, svel, rp, start, end, sp, s.fluid, s.common, s.kernels, s.key_mode,
                               v_out_init=s.vel, want_acc=True)
    _, _, mag = orc.forces(spos, svel, rp.astype(np.float64), start, end, sp, s.fluid, s.common, s.kernels,
                           s.key_mode, f64=True, want_mag=True)
    vel, _ = gpu_forces(fglib, s, spos, svel, rp, start, end, sp, abi.MATH_REFERENCE)
    check_velocity(vel, v_ref.astype(np.float64), acc, mag, sp, s.common.deltaTimeIntegration)
