"""The tile schedules of the electron diffusion against the group-by-group
sweep (tests/native/dte_plan_check.cpp): forward, backward and both sweeps,
bit for bit, over every mesh of the given sides."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "spilady_amd", "csrc")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("dte") / "dte_plan_check")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-pthread", "-I" + CSRC, "-o", exe,
                           os.path.join(HERE, "native", "dte_plan_check.cpp"),
                           os.path.join(CSRC, "sld_dte_plan.cpp")])
    return exe


# even and odd sides, sides below a tile, remainders of 1 to edge - 1
@pytest.mark.parametrize("lo,hi,edges", [(3, 9, (1, 4, 6)), (10, 13, (4, 8)), (17, 18, (4, 10)), (27, 27, (6,))])
def test_tiles_reproduce_the_sweeps(check, lo, hi, edges):
    out = subprocess.run([check, str(lo), str(hi), *map(str, edges)], capture_output=True, text=True)
    assert out.returncode == 0 and "bad 0" in out.stdout, out.stdout[-2000:]
