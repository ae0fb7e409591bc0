"""The host loops of the list generators on kept worker threads (csrc/parallel.hpp)."""
import os
import subprocess

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "plancheck")


def test_loops_on_kept_threads(tmp_path):
    exe = str(tmp_path / "pool_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", os.path.join(HERE, "pool_check.cpp"), "-o", exe], check=True, timeout=120)
    assert subprocess.run([exe], timeout=60).returncode == 0
