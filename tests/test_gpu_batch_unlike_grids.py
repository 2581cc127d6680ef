"""A batch whose scenes' grids differ strongly in size, small before large and
large before small, so that wavefronts at the scenes' boundaries span unlike
grids: every schedule gives the row schedule's bits, and the tuner, which
tries all of them, leaves the state as it was."""
import numpy as np
import pytest

from fluidgrid_amd import scenes

pytestmark = pytest.mark.gpu

SMALL, LARGE = ((12, 9, 8), 0.4), ((40, 20, 41), 1.9)  # particles per axis, box edge (8 and 38 cells)


def _batch(fglib, which):
    parts = []
    for k, (lattice, edge) in enumerate(which):
        s = scenes.dam_break(lattice, 0.05, (edge,) * 3, 1e-4, seed=k)
        s.vel[:, :3] = np.random.default_rng(k).normal(0.0, 0.2, (s.n, 3))
        parts.append(s)
    return fglib.BatchSimulator(scenes.Ensemble(parts, 0, None))


@pytest.mark.parametrize("which", [(SMALL, LARGE), (LARGE, SMALL), (SMALL, LARGE, SMALL, SMALL)],
                         ids=["small_large", "large_small", "four"])
def test_schedules_give_the_same_bits(fglib, which):
    want = None
    for flat_density, flat_forces in ((0, 0), (1, 0), (0, 1), (1, 1)):
        for block in (64, 256):
            b = _batch(fglib, which)
            try:
                b.set_tuning(block, 8, flat_density, flat_forces)
                b.step(3)
                got = np.stack(b.state())
            finally:
                b.close()
                fglib.load().fg_set_tuning(64, 8)
                fglib.load().fg_set_schedule(0, 0)
            want = got if want is None else want
            assert np.array_equal(got, want), (flat_density, flat_forces, block)


def test_tuner_leaves_the_state(fglib):
    b = _batch(fglib, (SMALL, LARGE))
    try:
        before = np.stack(b.state())
        b.autotune(trial_steps=2)
        assert np.array_equal(np.stack(b.state()), before)
    finally:
        b.close()
        fglib.load().fg_set_tuning(64, 8)
        fglib.load().fg_set_schedule(0, 0)
