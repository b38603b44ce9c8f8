"""The host's side of a PCG run's progress in pinned memory, on the CPU (tests/cpp/pcg_wait.cpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _run(tmp_path, what):
    exe = os.path.join(tmp_path, "pcg_wait")
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                           os.path.join(ROOT, "tests", "cpp", "pcg_wait.cpp"), "-pthread", "-o", exe])
    r = subprocess.run([exe, what], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip().endswith("OK"), r.stdout + r.stderr


def test_an_invalid_element_is_known_with_the_first_state(tmp_path):
    """The flag comes with the run's state, not from a copy that only a synchronisation makes readable."""
    _run(tmp_path, "flags")


def test_waits_share_a_core(tmp_path):
    """Threads that wait for their runs on one core give it to each other."""
    _run(tmp_path, "sharing")


def test_a_failed_run_ends_the_wait(tmp_path):
    _run(tmp_path, "failure")
