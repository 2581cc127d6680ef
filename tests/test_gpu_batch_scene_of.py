"""The scene of each particle, written on the GPU: scenes of one particle, of
none (first, between and last) and of more than a wavefront's give each
particle the bits it has in a batch of its scene alone."""
import dataclasses

import numpy as np
import pytest

from fluidgrid_amd import scenes

pytestmark = pytest.mark.gpu


def _run(fglib, parts):
    sim = fglib.BatchSimulator(scenes.Ensemble(parts, 0, None))
    try:
        sim.step(3)
        return np.stack(sim.state())
    finally:
        sim.close()


@pytest.mark.parametrize("counts", [(1,), (0, 1, 65, 0, 0, 300, 1, 0), (64, 128, 1, 63), (3, 0)])
def test_scene_boundaries(fglib, counts):
    parts = []
    for k, n in enumerate(counts):
        s = scenes.dam_break((8, 6, 8), 0.02, (1.0, 1.0, 1.0), 1e-4, seed=k)
        s.vel[:, :3] = np.random.default_rng(k).normal(0.0, 0.2, (s.n, 3))
        parts.append(dataclasses.replace(s, pos=s.pos[:n].copy(), vel=s.vel[:n].copy()))
    got = _run(fglib, parts)
    want = [_run(fglib, [p]) for p in parts if p.n]
    assert np.array_equal(got, np.concatenate(want, axis=1))
