"""The growth of the prompt chunks' scratch (pokitlms_amd/csrc/chunk_scratch.hpp)
under an allocator that fails: a short prompt, a long one that finds no memory, a
short one again.  The scratch must be a live block or empty after each."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_growth_and_failed_growth(tmp_path):
    exe = str(tmp_path / "chunk_scratch_cases")
    src = os.path.join(ROOT, "tests", "native", "chunk_scratch_cases.cpp")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", src, "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.count("PASS") == 3, r.stdout
