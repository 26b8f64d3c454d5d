"""What a solver keeps between batched solves: the FP32 coarse inverse follows the coefficients.

Tolerances: solves to 1e-8 of the same problem agree to 1e-6 (a residual reduced by 1e-8 times the
operator's condition on these meshes, below 100 after preconditioning).
"""
import numpy as np
import pytest

import dendro_amd as da
from tests.meshes import hierarchy, rel_err, var_coefficients

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

K = 8


@pytest.fixture(scope="module")
def hier():
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    da.init(0)
    return hierarchy("clusters", 6000, 10, 3, seed=4, min_coarse=50)


def build(h, scale=1.0, **kw):
    c = var_coefficients(h, mass_base=1.0)
    ms = []
    for l in range(h.n):
        m = da.Mesh(h.levels[l])
        m.set_coefficients(c[l][0] * scale, c[l][1] * scale)
        ms.append(m)
    ts = [da.Transfer(ms[l - 1], ms[l], *h.transfers[l - 1]) for l in range(1, h.n)]
    p = dict(omega=2.0 / 3.0, nu_pre=2, nu_post=2, rtol=1e-8, max_it=60, norm_type=da.NORM_UNPRECONDITIONED)
    p.update(kw)
    return ms, da.Solver(ms, ts, da.default_params(**p))


def rescale(h, ms, scale):
    c = var_coefficients(h, mass_base=1.0)
    for l, m in enumerate(ms):
        m.set_coefficients(c[l][0] * scale, c[l][1] * scale)


@pytest.mark.parametrize("prec", [da.F64, da.F32])
@pytest.mark.parametrize("graph", [0, 1])
def test_batched_solve_after_new_coefficients(hier, prec, graph):
    B = torch.tensor(np.random.default_rng(2).uniform(-1, 1, (hier.fine.n_node, K)), device="cuda:0")
    X, Y = torch.empty_like(B), torch.empty_like(B)
    ms, s = build(hier, vcycle_prec=prec, use_graph=graph)
    s.solve_multi(B, X, K)
    rescale(hier, ms, 64.0)
    got = s.solve_multi(B, X, K)
    ref = build(hier, 64.0, vcycle_prec=prec, use_graph=graph)[1].solve_multi(B, Y, K)
    assert all(st.converged for st in ref)
    assert [st.iterations for st in got] == [st.iterations for st in ref]
    assert rel_err(X.cpu().numpy(), Y.cpu().numpy()) <= 1e-6
