"""Which EAS meshes are staged in chunks, on the CPU (tests/cpp/pattern_chunks.cpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_chunks_by_size_and_numbering(tmp_path):
    """Equal chunks of about 131,072 elements where the numbering completes rows on the way, else one chunk; a given
    chunk size is taken as it is."""
    exe = os.path.join(tmp_path, "pattern_chunks")
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                           os.path.join(ROOT, "ikarus_amd", "csrc", "pattern.cpp"),
                           os.path.join(ROOT, "tests", "cpp", "pattern_chunks.cpp"), "-pthread", "-o", exe])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=200)
    assert r.returncode == 0 and r.stdout.strip().endswith("OK"), r.stdout + r.stderr
