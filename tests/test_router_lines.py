"""The line from the router's tiles of four by four to the matrix units (mummu_amd/csrc/router_lines.h), asked by a test program on the CPU: calls whose experts
would leave most of a matrix tile's columns empty stay with the former."""
import os
import subprocess

from mummu_amd import build


def test_matrix_units_only_for_columns_that_hold_experts(tmp_path):
    binary = str(tmp_path / "router_lines_test")
    subprocess.run([os.environ.get("CXX", "g++"), "-O1", "-std=c++17", "-Wall", "-I", os.path.join(build.HERE, "csrc"),
                    os.path.join(build.ROOT, "tests", "cpp", "router_lines_test.cpp"), "-o", binary], check=True, timeout=100)
    r = subprocess.run([binary], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "router lines: ok" in r.stdout
