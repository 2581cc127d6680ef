"""Rows that the density and force passes cannot stage as usual: more than 64
candidates a lane (no mask), more than 127 particles in three cells (ranges
looked up), runs that are long for what the lanes read of them or longer than
the longest (read from memory), next to ordinary ones in a wavefront, and
particles at non-finite positions.  The flat schedules, which stage nothing,
and the launchers without a neighbour buffer give the same bits; densities and
velocities are the FP32 oracle's with the tolerances of test_gpu_sph.py."""
import numpy as np
import pytest

from fluidgrid_amd import abi
from test_gpu_row_runs import H, _block, _scene
from test_gpu_sph import check_density, check_velocity, grid_cpu

pytestmark = pytest.mark.gpu


def _cells(s, cell):
    """The scene on cells of another size."""
    ext = [float(v) for v in s.common.volume_max]
    s.common.cell_size = abi.f3(cell, cell, cell)
    s.common.bucket_size = abi.i3(*[int(np.ceil(e / cell - 1e-6)) for e in ext])
    return s


def _three_cells(count):
    """`count` particles in three cells in a row, and few around them."""
    return _scene(np.concatenate([_block(count, (0.2, 0.2, 0.2), (0.35, 0.25, 0.25)), _block(200, 0.0, 0.6, 2)]))


def _pool_and_line(count):
    """A pool, and a few particles along a line of cells above it: a wavefront
    of them spans the line, and its runs in the rows below are `count` long."""
    x = np.linspace(0.0, 0.999, 70)
    line = np.stack([x, np.full(70, 0.105), np.full(70, 0.105)], 1)
    return _scene(np.concatenate([_block(count, (0.0, 0.05, 0.05), (0.999, 0.1, 0.1)), line, _block(300, 0.2, 0.999, 3)]))


def _not_finite():
    s = _scene(_block(3000, 0.1, 0.6))
    rng = np.random.default_rng(5)
    for value in (np.nan, np.inf, -np.inf, 3.2e38, -1e30):
        for axis in range(3):
            s.pos[rng.integers(0, s.n, 4), axis] = value
    return s


CASES = {
    "three_cells_64": lambda: _three_cells(64),
    "three_cells_65": lambda: _three_cells(65),
    "three_cells_127": lambda: _three_cells(127),
    "three_cells_128": lambda: _three_cells(128),
    "three_cells_700": lambda: _three_cells(700),
    "clump_2600": lambda: _scene(np.concatenate([_block(2600, 0.21, 0.24), _block(300, 0.0, 0.6, 2)])),
    "cells_of_2h": lambda: _cells(_scene(_block(9000, 0.0, (0.5, 0.4, 0.5))), 2 * H),
    "cells_of_3h": lambda: _cells(_scene(_block(9000, 0.0, (0.5, 0.4, 0.5))), 3 * H),
    "compressed": lambda: _scene(_block(9000, 0.0, (0.3, 0.25, 0.3))),
    "run_600": lambda: _pool_and_line(600),
    "run_700": lambda: _pool_and_line(700),
    "run_2040": lambda: _pool_and_line(2040),
    "run_2060": lambda: _pool_and_line(2060),
    "not_finite": _not_finite,
}


@pytest.mark.parametrize("which", list(CASES))
def test_schedules_and_oracle(fglib, orc, which):
    s = CASES[which]()
    L = fglib.load()
    _, sp, start, end, spos, svel = grid_cpu(orc, s)
    fglib.init_params(s.common, s.kernels, s.key_mode, abi.MATH_FAST)
    d = {k: fglib.DeviceArray.from_numpy(v) for k, v in dict(spos=spos, svel=svel, start=start, end=end, sp=sp).items()}
    nbr = fglib.DeviceArray((L.fg_neighbor_mask_bytes(s.n),), np.uint8)

    def run(flat_density, flat_forces, masks=True):
        rp = fglib.DeviceArray.from_numpy(np.zeros((s.n, 2), np.float32))
        vel = fglib.DeviceArray.from_numpy(s.vel)
        fglib.check(L.fg_set_schedule(flat_density, flat_forces))
        try:
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
            return rp.numpy().view(np.uint32), vel.numpy().view(np.uint32)
        finally:
            L.fg_set_schedule(0, 0)

    rp, vel = run(0, 0)
    for other in (run(1, 1), run(1, 0), run(0, 1), run(0, 0, False)):
        assert np.array_equal(other[0], rp) and np.array_equal(other[1], vel)
    if which == "not_finite":
        return
    rp, vel = rp.view(np.float32), vel.view(np.float32)
    check_density(rp, orc.density(spos, start, end, s.fluid, s.common, s.kernels, s.key_mode), s)
    v_ref, acc, _ = orc.forces(spos, svel, rp, start, end, sp, s.fluid, s.common, s.kernels, s.key_mode,
                               v_out_init=s.vel, want_acc=True)
    _, _, mag = orc.forces(spos, svel, rp.astype(np.float64), start, end, sp, s.fluid, s.common, s.kernels,
                           s.key_mode, f64=True, want_mag=True)
    check_velocity(vel, v_ref.astype(np.float64), acc, mag, sp, s.common.deltaTimeIntegration)


@pytest.mark.parametrize("which", [k for k in CASES if k != "not_finite"])
def test_mixed_precision_masks(fglib, orc, which):
    """The mixed-precision density pass on the same rows: the FP32 pass's masks
    bit for bit, and its densities within 4e-6: the roundings (2^-24 each) of
    the FP32 pass's plain sum, of up to some thousand terms in random order,
    whose square root they grow with; the compensated sum's are below them."""
    s = CASES[which]()
    L = fglib.load()
    sk, sp, start, end, spos, _ = grid_cpu(orc, s)
    fglib.init_params(s.common, s.kernels, s.key_mode, abi.MATH_FAST)
    d = {k: fglib.DeviceArray.from_numpy(v) for k, v in dict(key=sk, sp=sp, pos=s.pos, vel=s.vel).items()}
    nb = s.num_buckets
    out = []
    for precision in (abi.PRECISION_FP32, abi.PRECISION_MIXED):
        fglib.check(L.fg_set_precision(precision))
        try:
            g = {k: fglib.DeviceArray((nb,), np.uint32) for k in ("start", "end")}
            o = {k: fglib.DeviceArray((s.n, 4), np.float32) for k in ("pos", "vel")}
            rp = fglib.DeviceArray.from_numpy(np.zeros((s.n, 2), np.float32))
            nbr = fglib.DeviceArray((L.fg_neighbor_mask_bytes(s.n),), np.uint8)
            fglib.check(L.fg_cell_offsets_pos_vel(g["start"].ptr, g["end"].ptr, d["key"].ptr, d["sp"].ptr, d["pos"].ptr,
                                                  o["pos"].ptr, d["vel"].ptr, o["vel"].ptr, s.n, nb, 1, nbr.ptr))
            fglib.check(L.fg_sph_density_nbr(o["pos"].ptr, o["vel"].ptr, rp.ptr, g["start"].ptr, g["end"].ptr, nbr.ptr,
                                             s.n, s.fluid.gasConstant, s.fluid.restDensity, s.fluid.mass))
            assert np.array_equal(o["pos"].numpy(), spos)
            out.append((rp.numpy()[:, 0], fglib.download_raw(nbr.ptr, (9, s.n), np.uint64)))
        finally:
            L.fg_set_precision(abi.PRECISION_FP32)
    assert np.array_equal(out[0][1], out[1][1])
    assert np.all(np.abs(out[0][0] - out[1][0]) <= 4e-6 * out[0][0])
