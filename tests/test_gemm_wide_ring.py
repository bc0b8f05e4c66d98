"""The wide GEMM's stages in LDS and the loads that its waves count (mummu_amd/csrc/gemm_wide_ring.h), walked by a test program on the CPU: every stage is
asked for once and has landed before it is read, for tiles of every height behind every other."""
import os
import subprocess

from mummu_amd import build


def test_every_stage_is_asked_for_once_and_has_landed(tmp_path):
    binary = str(tmp_path / "gemm_wide_ring_test")
    subprocess.run([os.environ.get("CXX", "g++"), "-O1", "-std=c++17", "-Wall", "-I", os.path.join(build.HERE, "csrc"),
                    os.path.join(build.ROOT, "tests", "cpp", "gemm_wide_ring_test.cpp"), "-o", binary], check=True, timeout=100)
    r = subprocess.run([binary], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "wide ring: ok" in r.stdout
