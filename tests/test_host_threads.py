"""Host work shared among threads (spilady_amd/csrc/sld_threads.h) where a
thread or a thread's memory cannot be had (tests/native/host_threads_check.cpp):
the calling thread does the work to the same bits, and an allocation that fails
inside a thread is the caller's exception, not the end of the process."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "spilady_amd", "csrc")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("threads") / "host_threads_check")
    src = [os.path.join(CSRC, f) for f in ("sld_dte_plan.cpp", "sld_model.cpp", "sld_tables.cpp")]
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-pthread", "-I" + CSRC, "-o", exe,
                           os.path.join(HERE, "native", "host_threads_check.cpp"), *src, "-ldl"])
    return lambda mode: subprocess.run([exe, mode], capture_output=True, text=True, timeout=120)


def test_no_thread_to_be_had(check):
    a, b = check("threads"), check("none")
    assert a.returncode == 0, a.stderr
    assert b.returncode == 0, b.stderr
    assert a.stdout.count("\n") == 3 and b.stdout == a.stdout


@pytest.mark.skipif(len(os.sched_getaffinity(0)) < 2, reason="one processor: no thread is made")
def test_no_memory_inside_a_thread(check):
    r = check("memory")
    assert r.returncode == 0 and r.stdout == "bad_alloc in the caller\n", (r.returncode, r.stdout, r.stderr)
