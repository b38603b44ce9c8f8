"""What the numbering of a mesh decides, on the CPU (tests/cpp/pattern_chunks.cpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _run(tmp_path, *what):
    exe = os.path.join(tmp_path, "pattern_chunks")
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                           os.path.join(ROOT, "ikarus_amd", "csrc", "pattern.cpp"),
                           os.path.join(ROOT, "tests", "cpp", "pattern_chunks.cpp"), "-pthread", "-o", exe])
    r = subprocess.run([exe, *what], capture_output=True, text=True, timeout=200)
    assert r.returncode == 0 and r.stdout.strip().endswith("OK"), r.stdout + r.stderr


def test_chunks_by_size_and_numbering(tmp_path):
    """Equal chunks of about 131,072 elements where the numbering completes rows on the way, else one chunk; a given
    chunk size is taken as it is."""
    _run(tmp_path)


def test_stores_of_k_by_size_and_numbering(tmp_path):
    """How complete K blocks are stored: past the caches above the size of the last-level cache, but for Neo-Hooke far
    above it only where a tile's blocks do not follow each other in K."""
    _run(tmp_path, "stores")
