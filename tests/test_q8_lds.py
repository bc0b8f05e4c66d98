"""Where gemm_q8.hip reads rows in LDS (mummu_amd/csrc/gemm_q8_lds.h), driven by its own test program on the CPU: no read leaves the
workgroup's LDS, for items of either kind (up to 16 rows, more)."""
import os
import subprocess

from mummu_amd import build


def test_every_read_of_rows_stays_in_its_stage(tmp_path):
    binary = str(tmp_path / "q8_lds_test")
    subprocess.run([os.environ.get("CXX", "g++"), "-O1", "-std=c++17", "-Wall", "-I", os.path.join(build.HERE, "csrc"),
                    os.path.join(build.ROOT, "tests", "cpp", "q8_lds_test.cpp"), "-o", binary], check=True, timeout=100)
    r = subprocess.run([binary], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "q8 lds: ok" in r.stdout
