"""sld_model_set_params where the device has no memory left for one of its buffers
(tests/native/model_memory_check.cpp makes hipMalloc refuse on the host): an error,
and the next call, with the memory there, works. No kernel runs on what is missing."""
import os
import subprocess

import numpy as np
import pytest

from helpers import fe_params

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "spilady_amd")


def test_a_refused_buffer_is_an_error_and_no_more(tmp_path):
    v, p, at = fe_params(5, 300.0, 3, thermostats=False)
    state = tmp_path / "state"
    with open(state, "wb") as f:
        f.write(np.int32(at.natom).tobytes() + bytes(p))
        for k in ("r", "p", "s"):
            f.write(np.ascontiguousarray(getattr(at, k), dtype=np.float64).tobytes())
    exe = tmp_path / "model_memory_check"
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "include"), "-o", str(exe),
                           os.path.join(ROOT, "tests", "native", "model_memory_check.cpp"), "-L" + LIB,
                           "-lspilady_hip", "-Wl,-rpath," + LIB, "-ldl"])
    r = subprocess.run([str(exe), str(state)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
