"""Build-level guards with the library's own compiler flags (CPU: hipcc cross-compiles gfx950 assembly).

LDS: the operator, two-sweep and elasticity kernels address theirs from byte 0, which holds only while
they declare none of their own.  No kernel that runs per element spills.
Registers: default tilings run 1024-thread workgroups, two per CU, which needs at most 64 VGPRs; every
factored operator mode that takes them is held to that, the Dirichlet product among them."""
import os
import re
import shutil
import subprocess

import pytest

from dendro_amd import build as b


def _compile(tmp_path_factory, src):
    if not os.path.exists(b.HIPCC) and not shutil.which(b.HIPCC):
        pytest.skip("hipcc not available")
    out = str(tmp_path_factory.mktemp("asm") / (src + ".s"))
    r = subprocess.run([b.HIPCC] + b.HIP_FLAGS + ["-I" + os.path.join(b.ROOT, "include"), "-I" + b.CSRC, "--cuda-device-only",
                                                  "-S", os.path.join(b.CSRC, "device", src), "-o", out],
                       capture_output=True, text=True, timeout=900)
    assert r.returncode == 0, r.stderr[-2000:]
    return open(out).read()


@pytest.fixture(scope="module")
def asm(tmp_path_factory):
    return _compile(tmp_path_factory, "device_api.hip")


@pytest.fixture(scope="module")
def asm_elas(tmp_path_factory):
    return _compile(tmp_path_factory, "elas_api.hip")


@pytest.fixture(scope="module")
def asm_multi(tmp_path_factory):
    return _compile(tmp_path_factory, "multi_api.hip")


def _kernels(asm, pattern):
    ks = re.findall(r"\.amdhsa_kernel (\S+)\n(.*?)\.end_amdhsa_kernel", asm, re.S)
    return [(n, text) for n, text in ks if re.search(pattern, n)]


def _field(text, name):
    return int(re.search(r"\.amdhsa_%s (\d+)" % name, text).group(1))


def test_1024_thread_factored_kernels_fit_two_workgroups_per_cu(asm):
    """tile_op_kernel<T, T, MASS, MODE, 1024, UNI, false, false, true>, the product, residual, smoothing, CG
    and Dirichlet modes"""
    for mode in (0, 2, 3, 4, 5):
        ks = _kernels(asm, r"tile_op_kernel.*Li%dELi1024ELb[01]ELb0ELb0ELb1E" % mode)
        assert len(ks) >= 3, mode
        over = [(n, _field(t, "next_free_vgpr")) for n, t in ks if _field(t, "next_free_vgpr") > 64]
        assert not over, over


def _check(ks, at_least, own_lds=False):
    assert len(ks) >= at_least, len(ks)
    assert own_lds or not [n for n, t in ks if _field(t, "group_segment_fixed_size")]
    assert not [n for n, t in ks if _field(t, "private_segment_fixed_size")]


def test_fixed_lds_kernels_declare_none_and_do_not_spill(asm, asm_elas):
    _check(_kernels(asm, "tile_op_kernel"), 100)
    _check(_kernels(asm, "tile_pair_kernel"), 12)   # two precisions, two modes, three coefficient forms
    _check(_kernels(asm_elas, "elas_tile_kernel"), 1)


def test_batched_and_transfer_kernels_do_not_spill(asm, asm_multi):
    _check(_kernels(asm_multi, "tile_multi_kernel"), 40, own_lds=True)
    _check(_kernels(asm_multi, "dense_multi_kernel"), 2, own_lds=True)
    _check(_kernels(asm, "restrict_tile_kernel|prolong_tile_kernel"), 24, own_lds=True)


def test_every_hip_source_is_built_without_packed_fp32():
    i = b.HIP_FLAGS.index("-packed-fp32-ops")
    assert b.HIP_FLAGS[i - 3:i] == ["-Xclang", "-target-feature", "-Xclang"]
