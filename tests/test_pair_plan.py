"""The two-sweep tile plan (build_pair_tiles) against the contract its kernel relies on, checked on
the CPU by tests/pair_plan_check.cpp: tiles of one element, of ordinary sizes and of the whole mesh."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HOST = ["stencils.cpp", "octree.cpp", "da.cpp", "tiles.cpp", "host_api.cpp"]


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("pair") / "pair_plan_check")
    cmd = ["g++", "-O2", "-std=c++17", "-pthread", "-I" + os.path.join(ROOT, "include"),
           "-I" + os.path.join(ROOT, "dendro_amd", "csrc"), os.path.join(ROOT, "tests", "pair_plan_check.cpp"),
           *[os.path.join(ROOT, "dendro_amd", "csrc", "host", s) for s in HOST], "-o", out]
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr
    return out


@pytest.mark.parametrize("kind,npts,depth", [(0, 1, 3), (0, 3000, 6), (1, 2000, 9), (3, 1500, 10)])
def test_pair_plan_contract(checker, kind, npts, depth):
    r = subprocess.run([checker, str(kind), str(npts), str(depth)], capture_output=True, text=True, timeout=600)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
