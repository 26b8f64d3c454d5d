"""Host plans against the contracts their kernels rely on, checked on the CPU: the two-sweep tiles
(build_pair_tiles, tests/pair_plan_check.cpp) with tiles of one element, of ordinary sizes and of the
whole mesh, and the transfers' gather blocks (build_gather, tests/gather_plan_check.cpp)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HOST = ["stencils.cpp", "octree.cpp", "da.cpp", "tiles.cpp", "host_api.cpp"]


def _compile(tmp_path_factory, name):
    out = str(tmp_path_factory.mktemp("plan") / name)
    cmd = ["g++", "-O2", "-std=c++17", "-pthread", "-I" + os.path.join(ROOT, "include"),
           "-I" + os.path.join(ROOT, "dendro_amd", "csrc"), os.path.join(ROOT, "tests", name + ".cpp"),
           *[os.path.join(ROOT, "dendro_amd", "csrc", "host", s) for s in HOST], "-o", out]
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr
    return out


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    return _compile(tmp_path_factory, "pair_plan_check")


@pytest.mark.parametrize("kind,npts,depth", [(0, 1, 3), (0, 3000, 6), (1, 2000, 9), (3, 1500, 10)])
def test_pair_plan_contract(checker, kind, npts, depth):
    r = subprocess.run([checker, str(kind), str(npts), str(depth)], capture_output=True, text=True, timeout=600)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr


def test_gather_plan_contract(tmp_path_factory):
    r = subprocess.run([_compile(tmp_path_factory, "gather_plan_check")], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stdout + r.stderr
