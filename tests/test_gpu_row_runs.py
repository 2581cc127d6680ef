"""The density and force passes that stage each stencil row's run per
wavefront (fg_sph_density_nbr, then fg_sph_forces_integrate_nbr), where the
runs can go wrong, against the FP32 oracle with the tolerances of
test_gpu_sph.py (stated there per quantity), and the row masks against a
brute-force test of the same FP32 distances."""
import numpy as np
import pytest

from fluidgrid_amd import abi, scenes
from test_gpu_sph import check_density, check_velocity, grid_cpu

pytestmark = pytest.mark.gpu

H = 0.05


def _scene(pos, box=(1.0, 1.0, 1.0), scale=1.0):
    s = scenes.dam_break((2, 2, 2), H, box, 4e-4)
    rng = np.random.default_rng(len(pos))
    s.pos = np.ones((len(pos), 4), np.float32)
    s.pos[:, :3] = pos
    s.vel = np.zeros((len(pos), 4), np.float32)
    s.vel[:, :3] = rng.normal(0.0, 0.3, (len(pos), 3))
    s.fluid.max_particles = len(pos)
    if scale != 1.0:  # h and the cells in world units: h^2 / s^2 and (h / s)^2 then round apart
        s.common.simulation_scale = scale
        hw = np.float32(H) / np.float32(scale)
        s.pos[:, :3] /= np.float32(scale)
        s.common.cell_size = abi.f3(hw, hw, hw)
        s.common.volume_max = abi.f3(*[b / scale for b in box])
    return s


def _block(n, lo, hi, seed=1):
    return np.random.default_rng(seed).uniform(lo, hi, (n, 3))


CASES = {
    # one wavefront, one lane more, one less: without and with the runs table
    "n63": lambda: _scene(_block(63, 0.1, 0.25)),
    "n64": lambda: _scene(_block(64, 0.1, 0.25)),
    "n65": lambda: _scene(_block(65, 0.1, 0.25)),
    # a sparse layer on a dense one: wavefronts over many cells, whose runs in the row below fill
    # the staged slices more than once, and rows of more than 32 candidates
    "sparse_on_dense": lambda: _scene(np.concatenate([_block(6000, (0.0, 0.0, 0.0), (0.95, 0.2, 0.2)),
                                                      _block(260, (0.0, 0.0, 0.2), (0.95, 0.25, 0.25), 2)])),
    # particles far apart between dense clumps: runs longer than the longest
    "spray": lambda: _scene(np.concatenate([_block(5000, (0.3, 0.0, 0.3), (0.7, 0.15, 0.6)),
                                            _block(300, 0.0, 0.99, 3)])),
    # three cells with more than 64 and more than 127 particles
    "rows_over_64": lambda: _scene(_block(2500, 0.2, 0.4)),
    "rows_over_127": lambda: _scene(_block(2500, 0.2, 0.32)),
    # grids one, two and three cells wide: a row's next keys are the next row's cells
    "narrow_1": lambda: _scene(_block(700, 0.0, (0.05, 0.5, 0.5)), (0.05, 1.0, 1.0)),
    "narrow_2": lambda: _scene(_block(1200, 0.0, (0.1, 0.5, 0.5)), (0.1, 1.0, 1.0)),
    "narrow_3": lambda: _scene(_block(1500, 0.0, (0.15, 0.5, 0.5)), (0.15, 1.0, 1.0)),
    # particles outside the box, whose cells are clamped
    "outside": lambda: _scene(_block(3000, -0.15, 0.4)),
    "scaled": lambda: _scene(_block(3000, 0.1, 0.6), scale=0.009),
}


def _neighbours(spos, h, s):
    """|x_i - x_j|^2 < (h/s)^2 in the passes' FP32 operations, as a matrix."""
    f = np.float32
    x = spos[:, :3]
    d = x[:, None, :] - x[None, :, :]
    # one rounding per fused multiply-add, from exact products
    r2 = (d[..., 0] * d[..., 0]).astype(f)
    for k in (1, 2):
        r2 = (d[..., k].astype(np.float64) ** 2 + r2.astype(np.float64)).astype(f)
    hu = f(f(h) / f(s))
    return r2 < f(hu * hu)


def _long_rows(sk, dims):
    """Particles (sorted) with a stencil row whose three cells hold more than
    64 particles: such a row may have no mask."""
    count = np.bincount(sk, minlength=dims[0] * dims[1] * dims[2]).reshape(dims[2], dims[1], dims[0])
    c = np.pad(count, 1)
    row = c[:, :, :-2] + c[:, :, 1:-1] + c[:, :, 2:]
    most = np.max([row[1 + dz:1 + dz + dims[2], 1 + dy:1 + dy + dims[1]] for dz in (-1, 0, 1) for dy in (-1, 0, 1)], 0)
    return most.ravel()[sk] > 64


@pytest.mark.parametrize("which", list(CASES))
def test_runs_match_oracle(fglib, orc, which):
    s = CASES[which]()
    L = fglib.load()
    sk, sp, start, end, spos, svel = grid_cpu(orc, s)
    ref_rp = orc.density(spos, start, end, s.fluid, s.common, s.kernels, s.key_mode)
    fglib.init_params(s.common, s.kernels, s.key_mode, abi.MATH_FAST)
    d = {k: fglib.DeviceArray.from_numpy(v) for k, v in dict(spos=spos, svel=svel, start=start, end=end, sp=sp,
                                                             rp=np.zeros((s.n, 2), np.float32), vel=s.vel).items()}
    nbr = fglib.DeviceArray((L.fg_neighbor_mask_bytes(s.n),), np.uint8)
    fglib.check(L.fg_sph_density_nbr(d["spos"].ptr, d["svel"].ptr, d["rp"].ptr, d["start"].ptr, d["end"].ptr, nbr.ptr,
                                     s.n, s.fluid.gasConstant, s.fluid.restDensity, s.fluid.mass), "density")
    rp = d["rp"].numpy()
    check_density(rp, ref_rp, s)
    masks = fglib.download_raw(nbr.ptr, (9, s.n), np.uint64)
    near = _neighbours(spos, s.common.kernel_radius, s.common.simulation_scale).sum(1)
    bits = np.array([bin(int(v)).count("1") for v in masks.ravel()]).reshape(9, s.n).sum(0)
    long = _long_rows(sk, tuple(s.common.bucket_size))
    assert np.all(bits <= near) and np.array_equal(bits[~long], near[~long])
    v_ref, acc, _ = orc.forces(spos, svel, rp, start, end, sp, s.fluid, s.common, s.kernels, s.key_mode,
                               v_out_init=s.vel, want_acc=True)
    _, _, mag = orc.forces(spos, svel, rp.astype(np.float64), start, end, sp, s.fluid, s.common, s.kernels,
                           s.key_mode, f64=True, want_mag=True)
    fglib.check(L.fg_sph_forces_integrate_nbr(d["spos"].ptr, d["svel"].ptr, d["rp"].ptr, d["start"].ptr, d["end"].ptr,
                                              nbr.ptr, d["vel"].ptr, None, d["sp"].ptr, s.n, s.fluid.mass,
                                              s.fluid.viscosity), "forces")
    check_velocity(d["vel"].numpy(), v_ref.astype(np.float64), acc, mag, sp, s.common.deltaTimeIntegration)


@pytest.mark.parametrize("which", list(CASES))
def test_launchers_without_masks_give_the_same_bits(fglib, orc, which):
    """gCalcMassDensity and gSPHCalculateForces, which keep no neighbour
    buffer, against the passes that do: the same densities and velocities,
    bit for bit."""
    s = CASES[which]()
    L = fglib.load()
    sk, sp, start, end, spos, svel = grid_cpu(orc, s)
    fglib.init_params(s.common, s.kernels, s.key_mode, abi.MATH_FAST)
    d = {k: fglib.DeviceArray.from_numpy(v) for k, v in dict(spos=spos, svel=svel, start=start, end=end, sp=sp).items()}
    nbr = fglib.DeviceArray((L.fg_neighbor_mask_bytes(s.n),), np.uint8)
    out = []
    for masks in (True, False):
        rp = fglib.DeviceArray.from_numpy(np.zeros((s.n, 2), np.float32))
        vel = fglib.DeviceArray.from_numpy(s.vel)
        if masks:
            fglib.check(L.fg_sph_density_nbr(d["spos"].ptr, d["svel"].ptr, rp.ptr, d["start"].ptr, d["end"].ptr,
                                             nbr.ptr, s.n, s.fluid.gasConstant, s.fluid.restDensity, s.fluid.mass))
            fglib.check(L.fg_sph_forces_integrate_nbr(d["spos"].ptr, d["svel"].ptr, rp.ptr, d["start"].ptr,
                                                      d["end"].ptr, nbr.ptr, vel.ptr, None, d["sp"].ptr, s.n,
                                                      s.fluid.mass, s.fluid.viscosity))
        else:
            L.gCalcMassDensity(d["spos"].ptr, rp.ptr, None, d["start"].ptr, d["end"].ptr, s.n, s.fluid.gasConstant,
                               s.fluid.restDensity, s.fluid.mass)
            L.gSPHCalculateForces(d["spos"].ptr, d["svel"].ptr, None, rp.ptr, d["start"].ptr, d["end"].ptr, vel.ptr,
                                  d["sp"].ptr, s.n, s.fluid.mass, s.fluid.viscosity)
            fglib.check(None, "launchers")
        out.append((rp.numpy(), vel.numpy()))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
