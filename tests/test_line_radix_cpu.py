"""The plans of the line transforms take small radices wherever those fit (run on the
CPU from line_plan.h)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_small_radices_first(tmp_path):
    exe = str(tmp_path / "line_radix_check")
    subprocess.run(["g++", "-O1", "-std=c++17",
                    os.path.join(ROOT, "tests", "native", "line_radix_check.cpp"), "-o", exe],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
