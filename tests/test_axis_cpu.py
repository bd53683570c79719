"""The column arithmetic of whole runs (csrc/owm_axis.h, shared by host and
device) against direct compares with every window and cell edge."""
import os
import re
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_columns_equal_direct_compares(tmp_path):
    exe = str(tmp_path / "axis_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-o", exe,
                    os.path.join(HERE, "axis_check.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    n = [int(v) for v in re.findall(r"\d+", r.stdout)]
    assert r.returncode == 0, r.stdout
    # the draw reaches every path: certain and uncertain estimates, points
    # without a column, paired and unpaired grids
    assert n[0] > 1_000_000 and 0 < n[1] < n[0] and n[2] > 10_000 and 0 < n[3] < 4000
