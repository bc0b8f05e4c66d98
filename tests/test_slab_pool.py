"""The pool of pinned slabs (mummu_amd/csrc/slab_pool.h), driven by its own test program on the CPU: as many calls side by
side as there are handles allocate nothing once each has had a slab."""
import os
import subprocess

from mummu_amd import build


def test_calls_side_by_side_allocate_nothing_after_the_first_round(tmp_path):
    binary = str(tmp_path / "slab_pool_test")
    subprocess.run([os.environ.get("CXX", "g++"), "-O1", "-std=c++17", "-Wall", "-pthread", "-I", os.path.join(build.HERE, "csrc"),
                    os.path.join(build.ROOT, "tests", "cpp", "slab_pool_test.cpp"), "-o", binary], check=True, timeout=100)
    r = subprocess.run([binary], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "slab pool: ok" in r.stdout
