"""Restriction and prolongation through LDS blocks against the oracle: meshes of a few nodes, partial
last blocks, and a coarse level large enough for the two-lane restriction; onto another vector,
in place, and without an input vector; twice with equal bits.

Tolerances: each result is a sum of at most 64 products with weights that are exact in FP32, so
64 2^-53 and 64 2^-24 of the sum of absolute terms, which is at most a few times the result's norm
for random vectors: 1e-13 and 1e-5.
"""
import numpy as np
import pytest

import dendro_amd as da
import oracle
from tests.meshes import hierarchy, rel_err

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("mesh", [("uniform", 9, 4), ("clusters", 60, 7), ("lognormal", 900, 8), ("clusters", 9000, 10),
                                  ("lognormal", 250000, 11)])
def test_transfer_blocks(mesh):
    da.init(0)
    h = hierarchy(*mesh, 2, seed=3, min_coarse=1)
    C, F = h.levels
    ms = [da.Mesh(L) for L in h.levels]
    t = da.Transfer(ms[0], ms[1], *h.transfers[0])
    print(mesh, "coarse nodes", C.n_node, "fine nodes", F.n_node)
    assert mesh[1] < 250000 or C.n_node >= 80000
    rng = np.random.default_rng(9)
    f, c, x = rng.uniform(-1, 1, F.n_node), rng.uniform(-1, 1, C.n_node), rng.uniform(-1, 1, F.n_node)
    for prec, dt, tol in ((da.F64, torch.float64, 1e-13), (da.F32, torch.float32, 1e-5)):
        up = lambda a: torch.tensor(a, dtype=dt, device="cuda:0")
        ft, ct, xt = up(f), up(c), up(x)
        fr, cr, xr = (v.double().cpu().numpy() for v in (ft, ct, xt))
        out, again = torch.empty_like(ct), torch.empty_like(ct)
        t.restrict(ft, out, prec=prec)
        t.restrict(ft, again, prec=prec)
        assert torch.equal(out, again)
        assert rel_err(out.cpu().numpy(), oracle.restrict(C, F, fr)) <= tol
        pc = oracle.prolong(C, F, cr)
        y = torch.empty_like(xt)
        t.prolong_add(ct, xt, y, prec=prec)
        assert rel_err(y.cpu().numpy(), xr + pc) <= tol
        t.prolong_add(ct, xt, xt, prec=prec)
        assert torch.equal(xt, y)
        t.prolong_add(ct, None, y, prec=prec)
        assert rel_err(y.cpu().numpy(), pc) <= tol
