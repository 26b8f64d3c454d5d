"""Operator tilings of meshes whose elements are in random order (tests/shuffled_tiles_check.cpp), on the
CPU: accepted at every tile size, default ones among them, and within the kernels' capacities."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HOST = ["stencils.cpp", "octree.cpp", "da.cpp", "tiles.cpp", "host_api.cpp"]


def test_shuffled_tiles(tmp_path):
    out = str(tmp_path / "shuffled_tiles_check")
    r = subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-I" + os.path.join(ROOT, "include"),
                        "-I" + os.path.join(ROOT, "dendro_amd", "csrc"), os.path.join(ROOT, "tests", "shuffled_tiles_check.cpp"),
                        *[os.path.join(ROOT, "dendro_amd", "csrc", "host", s) for s in HOST], "-o", out],
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([out], capture_output=True, text=True, timeout=600)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
