"""The host planners under failing thread starts and allocations (tests/workers_check.cpp), on the CPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HOST = ["stencils.cpp", "octree.cpp", "da.cpp", "tiles.cpp", "host_api.cpp"]


def test_planners_without_threads_or_memory(tmp_path):
    out = str(tmp_path / "workers_check")
    r = subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-I" + os.path.join(ROOT, "include"),
                        "-I" + os.path.join(ROOT, "dendro_amd", "csrc"), os.path.join(ROOT, "tests", "workers_check.cpp"),
                        *[os.path.join(ROOT, "dendro_amd", "csrc", "host", s) for s in HOST], "-ldl", "-o", out],
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([out], capture_output=True, text=True, timeout=600)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
