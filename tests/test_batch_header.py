"""The batch simulator's C++ header: scenes given as lists in braces name the
vector of BatchScene, also an empty list and a scene without particles, and
vectors of both kinds are accepted (compiled, not run)."""
import os
import shutil
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CALLER = """
#include <fluidgrid/BatchedSimulator.h>
using namespace Simulation::Simulators;
void calls(const Simulation::Application::CommonFluidParams& c, const Simulation::Application::FluidParams& f,
           const std::vector<BatchScene>& s, const std::vector<BatchSceneView>& v) {
    BatchedSimulator none({}), list({s[0], s[1]}), bare({{c, f, {}, {}}}), scenes(s), views(v);
}
"""


def test_constructors_compile(tmp_path):
    src = tmp_path / "caller.cpp"
    src.write_text(CALLER)
    r = subprocess.run([shutil.which("g++"), "-std=c++17", "-fsyntax-only", "-w", "-D__HIP_PLATFORM_AMD__",
                        "-I", os.path.join(ROOT, "include"),
                        "-I", os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include"), str(src)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
