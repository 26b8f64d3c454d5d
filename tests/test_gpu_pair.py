"""Two smoothing sweeps per launch on small meshes: V-cycles against the oracle's for every split of
the sweeps into pairs and singles, each coefficient form, uniform and per element, meshes from a few
elements (one tile, most of its threads idle) to several hundred tiles, and after a change of
coefficients.

Tolerances: an FP64 V-cycle differs from the oracle's by rounding (1e-10, the bar of every V-cycle
here); an FP32 one by a few times 2^-24 per sweep and level, amplified by the smoothing operator's
condition (at most 4 levels, 8 sweeps: 1e-4).
"""
import numpy as np
import pytest

import dendro_amd as da
import oracle
from tests.meshes import hierarchy, rel_err, var_coefficients

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

MESHES = {"tiny": ("uniform", 9, 4, 2), "few": ("clusters", 60, 7, 2), "small": ("lognormal", 900, 8, 3),
          "tiles": ("clusters", 3000, 10, 3)}


@pytest.mark.parametrize("coef", ["uniform", "kappa", "kappa_mass"])
@pytest.mark.parametrize("mesh", sorted(MESHES))
def test_vcycle_of_pairs(mesh, coef):
    da.init(0)
    h = hierarchy(*MESHES[mesh], seed=3, min_coarse=1)
    assert h.n >= 2 and h.fine.n_elem < 60000
    ns = coef == "kappa"
    coefs = [(None, None)] * h.n if coef == "uniform" else var_coefficients(h, mass_base=None if ns else 1.0)
    ms = []
    for l in range(h.n):
        m = da.Mesh(h.levels[l])
        m.set_coefficients(*coefs[l])
        ms.append(m)
    ts = [da.Transfer(ms[l - 1], ms[l], *h.transfers[l - 1]) for l in range(1, h.n)]
    r = np.random.default_rng(5).uniform(-1, 1, h.fine.n_node)
    r -= r.mean() if ns else 0.0
    rt = torch.tensor(r, dtype=torch.float64, device="cuda:0")
    z = torch.empty_like(rt)

    def check(scale):
        lv = [(h.levels[l], None if k is None else k * scale, m if m is None else m * scale, scale, scale)
              for l, (k, m) in enumerate(coefs)]
        for pre, post in ((1, 1), (2, 2), (3, 3), (4, 1), (1, 4)):
            mg = oracle.MG(lv, omega=2.0 / 3.0, nu_pre=pre, nu_post=post, null_space=ns)
            ref = mg.vcycle(r)
            for prec, tol in ((da.F64, 1e-10), (da.F32, 1e-4)):
                s = da.Solver(ms, ts, da.default_params(omega=2.0 / 3.0, nu_pre=pre, nu_post=post, null_space=int(ns),
                                                        vcycle_prec=prec))
                s.vcycle(rt, z)
                e = rel_err(z.cpu().numpy(), ref)
                print(f"{mesh} {coef} scale {scale} nu {pre},{post} prec {prec}: {e:.2e}")
                assert e <= tol
                same = rt.clone()   # in place: the result may not be written while r is still read
                s.vcycle(same, same)
                assert torch.equal(same, z)

    check(1.0)
    for l, m in enumerate(ms):
        k, q = coefs[l]
        m.set_coefficients(None if k is None else k * 4.0, None if q is None else q * 4.0, 4.0, 4.0)
    check(4.0)
