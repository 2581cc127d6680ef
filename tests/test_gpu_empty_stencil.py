"""Cell-size relations with a negative axis, on which the reference's stencil
loops run no round (K_DeviceFunctions.cu:113-159): no body contact, whichever
and how many axes are negative, in the coupled launcher (both arithmetics)
and in the body forces."""
import numpy as np
import pytest

from fluidgrid_amd import abi
from test_gpu_boundary import _dev, _grids, _scene

pytestmark = pytest.mark.gpu

EMPTY = [(-1, 1, 1), (-1, -1, 1), (1, -2, -1), (-1, -1, -1)]


@pytest.mark.parametrize("math", [abi.MATH_FAST, abi.MATH_REFERENCE], ids=["fast", "reference"])
def test_coupled_launcher(fglib, orc, math):
    L = fglib.load()
    s, b = _scene()
    fglib.init_params(s.common, s.kernels, s.key_mode, math)
    g = _grids(orc, s, b)
    rp = orc.density(g["spos"], g["start"], g["end"], s.fluid, s.common, s.kernels, s.key_mode)
    d = {k: _dev(fglib, v) for k, v in dict(spos=g["spos"], svel=g["svel"], start=g["start"], end=g["end"], sp=g["sp"],
                                           rp=rp, bpos=g["bpos"], bvel=np.array([[0.05, -0.3, 0.02, 0.0]], np.float32),
                                           bstart=g["bstart"], bend=g["bend"]).items()}

    def velocities(relation):
        vel = _dev(fglib, s.vel)
        L.gSPHCalculateForcesWithSRB(
            d["spos"].ptr, d["svel"].ptr, None, vel.ptr, d["rp"].ptr, d["sp"].ptr, d["start"].ptr, d["end"].ptr, s.n,
            s.fluid.mass, s.fluid.viscosity, b.fluid_radius, abi.Int3(*relation), b.sphere_radius,
            abi.Float3(g["cell"], g["cell"], g["cell"]), -b.spring, -b.damping, None, None, None, 0, d["bpos"].ptr,
            d["bvel"].ptr, d["bstart"].ptr, d["bend"].ptr, g["nbb"], False, True)
        fglib.check(None, "gSPHCalculateForcesWithSRB")
        return vel.numpy()

    try:
        none = velocities((-1, 1, 1))
        assert not np.array_equal(velocities((1, 1, 1)), none)
        for relation in EMPTY:
            assert np.array_equal(velocities(relation), none), relation
    finally:
        fglib.init_params(s.common, s.kernels, s.key_mode, abi.MATH_FAST)


@pytest.mark.parametrize("relation", EMPTY)
def test_body_forces(fglib, orc, relation):
    L = fglib.load()
    s, b = _scene()
    fglib.init_params(s.common, s.kernels, s.key_mode)
    g = _grids(orc, s, b)
    cm = np.array([[*b.world[:, :3].mean(0), 0.0]], np.float32)
    d = {k: _dev(fglib, v) for k, v in dict(w=b.world, bv=np.zeros((1, 4), np.float32), cm=cm, spos=g["spos"],
                                           svel=g["svel"], start=g["start"], end=g["end"]).items()}
    f, t = fglib.DeviceArray((b.m, 4), np.float32), fglib.DeviceArray((b.m, 4), np.float32)
    fglib.check(L.fg_body_forces_from_fluid(d["w"].ptr, d["bv"].ptr, d["cm"].ptr, f.ptr, t.ptr, b.m, 1,
                                            b.sphere_radius, d["spos"].ptr, d["svel"].ptr, d["start"].ptr,
                                            d["end"].ptr, s.n, b.fluid_radius, abi.Float3(*s.common.cell_size),
                                            s.num_buckets, abi.Int3(*relation), -b.spring, -b.damping), "forces")
    assert not f.numpy()[:, :3].any() and not t.numpy()[:, :3].any()
