"""The segments of the Heff tiles' output blocks (csrc/segments.hpp) against the partial sums that
the product without allocation holds."""
import os
import subprocess

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "plancheck")


def test_segments_fit_the_product_without_allocation(tmp_path):
    exe = str(tmp_path / "segments_check")
    subprocess.run(["g++", "-O2", "-std=c++17", os.path.join(HERE, "segments_check.cpp"), "-o", exe], check=True, timeout=120)
    r = subprocess.run([exe], timeout=60, capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
