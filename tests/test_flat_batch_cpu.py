"""The flat density schedule over a batch whose scenes have unlike grids, as
its kernel runs on the CPU (cpu_wave/): no lookup leaves the cell tables, and
every particle has its own scene's density."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def build(tmp, name):
    """cpu_wave/<name>.cpp with the library's device code, as a CPU program."""
    out = os.path.join(str(tmp), name)
    rocm = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include")
    r = subprocess.run([shutil.which("g++"), "-std=c++20", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-ffp-contract=off",
                        "-I", os.path.join(ROOT, "tests", "cpu_wave"), "-I", os.path.join(ROOT, "include"),
                        "-I", os.path.join(ROOT, "fluidgrid_amd", "csrc"), "-I", rocm,
                        os.path.join(ROOT, "tests", "cpu_wave", name + ".cpp"), "-o", out], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return out


@pytest.fixture(scope="module")
def flat_batch(tmp_path_factory):
    return build(tmp_path_factory.mktemp("cpu_wave"), "flat_batch")


@pytest.mark.parametrize("scenes", [("8,100", "38,100"), ("38,100", "8,100"), ("3,70", "60,30", "3,70"),
                                    ("10,300", "10,300"), ("1,5", "40,200", "2,64", "5,3")])
def test_lookups_stay_in_the_tables(flat_batch, scenes):
    r = subprocess.run([flat_batch, *scenes], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.startswith("ok"), (r.returncode, r.stdout, r.stderr)
