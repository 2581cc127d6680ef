"""The launch of the mesh winding lattice (cpu_wave/): every lattice that the
entry point accepts, up to 2^34 points, fits a launch (fewer than 2^32 lanes
in x, at most 65,535 workgroups in y) and is covered by it, 128 points a
workgroup."""
import subprocess

import pytest

from test_flat_batch_cpu import build


@pytest.fixture(scope="module")
def mesh_launch(tmp_path_factory):
    return build(tmp_path_factory.mktemp("cpu_wave"), "mesh_launch")


@pytest.mark.parametrize("dims", [(1, 1, 1), (3, 5, 7), (812, 812, 812), (813, 813, 813), (1, 1 << 14, 1 << 14),
                                  (1, (1 << 14) + 1, 1 << 14), (1 << 11, 1 << 11, 1 << 11), (1 << 12, 1 << 11, 1 << 11),
                                  (1, 1 << 17, 1 << 17), (1 << 31, 8, 1), ((1 << 17) - 1, 1, 1 << 17)])
def test_every_lattice_fits(mesh_launch, dims):
    r = subprocess.run([mesh_launch, *map(str, dims)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.returncode
    x, y, lanes = map(int, r.stdout.split())
    assert x * lanes < 1 << 32 and 1 <= y <= 65535
    pairs = (dims[0] + 1) // 2 * dims[1] * dims[2]  # two neighbours of a row a lane
    assert x * y * 64 >= pairs
