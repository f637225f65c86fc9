"""The process keeps the bridge polynomials of a few cutoffs, not of every one it
has seen (tests/native/model_bridge_check.cpp)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "spilady_amd", "csrc")


def test_the_last_few_cutoffs_stay(tmp_path):
    exe = str(tmp_path / "model_bridge_check")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-pthread", "-I" + CSRC, "-o", exe,
                           os.path.join(HERE, "native", "model_bridge_check.cpp"),
                           os.path.join(CSRC, "sld_model.cpp"), os.path.join(CSRC, "sld_tables.cpp")])
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout == "alive 4 first 1 last 1\n", (out.returncode, out.stdout)
