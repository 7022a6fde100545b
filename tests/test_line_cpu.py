"""The plans of the fast line transforms (line_plan.h) for every length up to 514,
run on the CPU with the kernels' register DFTs against direct sums in long double.
Bound 5e-15 of the largest result: at most 5 passes, each with a product and a DFT
of at most 13 points, leave under 5 x 8 roundings of 1.1e-16."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_every_line_plan(tmp_path):
    exe = str(tmp_path / "line_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wno-unknown-pragmas",
                    os.path.join(ROOT, "tests", "native", "line_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
