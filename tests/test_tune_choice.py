"""The autotuner's choice among measured candidates (gpuvoxels_amd/csrc/vx3h_tune.h), on the
CPU: a workgroup size of its own only with a lead that no two runs of one configuration have."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpuvoxels_amd", "csrc")
SRC = """#include <cstdio>
#include "%s/vx3h_tune.h"
int main() {
    std::vector<vx3h_tune_trial> t;
    vx3h_tune_trial x{};
    while (scanf("%%d %%lf", &x.block_size, &x.voxel_steps_per_s) == 2) t.push_back(x);
    printf("%%zu", vx3::chooseTrial(t));
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    d = tmp_path_factory.mktemp("tune")
    (d / "choice.cpp").write_text(SRC % CSRC)
    subprocess.run(["g++", "-std=c++17", "-o", str(d / "choice"), str(d / "choice.cpp")], check=True)
    return str(d / "choice")


@pytest.mark.parametrize("trials,want", [
    ([(0, 13.377e9), (0, 13.2e9), (512, 13.389e9)], 0),      # a lead of 0.1%
    ([(0, 9.0e9), (0, 13.0e9), (256, 13.2e9)], 1),
    ([(0, 10.0e9), (256, 10.3e9), (512, 11.0e9)], 2),
    ([(256, 5.0), (512, 4.0)], 0),
    ([(512, 4.0), (0, 5.0), (0, 5.0)], 1),
    ([(0, 0.0), (128, 0.0)], 0)])
def test_choice(program, trials, want):
    out = subprocess.run([program], input="\n".join("%d %r" % t for t in trials), stdout=subprocess.PIPE, text=True, check=True).stdout
    assert int(out) == want
