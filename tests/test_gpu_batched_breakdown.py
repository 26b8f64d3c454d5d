"""Batched solves with a right-hand side that is not finite: reported as the single solve reports it, and
the other columns are solved to the same bits as without it.
"""
import numpy as np
import pytest

import dendro_amd as da
from dendro_amd import core
from tests.meshes import hierarchy, var_coefficients

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

K = 8


@pytest.mark.parametrize("norm", [da.NORM_UNPRECONDITIONED, da.NORM_PRECONDITIONED])
@pytest.mark.parametrize("columns", [[5], [0, 7], list(range(K))])
def test_nan_columns_are_reported(norm, columns):
    da.init(0)
    h = hierarchy("clusters", 6000, 10, 3, seed=4, min_coarse=50)
    ms = []
    for L, c in zip(h.levels, var_coefficients(h, mass_base=1.0)):
        m = da.Mesh(L)
        m.set_coefficients(*c)
        ms.append(m)
    ts = [da.Transfer(ms[l - 1], ms[l], *h.transfers[l - 1]) for l in range(1, h.n)]
    s = da.Solver(ms, ts, da.default_params(omega=2.0 / 3.0, nu_pre=2, nu_post=2, rtol=1e-8, max_it=60, norm_type=norm,
                                            vcycle_prec=da.F32))
    B = np.random.default_rng(2).uniform(-1, 1, (h.fine.n_node, K))
    B[:, columns] = 0.0
    Bt = torch.tensor(B, device="cuda:0")
    X, Y = torch.empty_like(Bt), torch.empty_like(Bt)
    ref = s.solve_multi(Bt, X, K)
    Bt[7, columns] = float("nan")
    with pytest.raises(da.DendroError):
        s.solve(Bt[:, columns[0]].contiguous(), torch.empty_like(Bt[:, 0]))
    st = (core.SolveStats * K)()
    rc = core.lib().dgh_solver_solve_multi(s.h, K, core.ptr(Bt), core.ptr(Y), st, None)
    assert rc < 0
    for j in range(K):
        if j in columns:
            assert not st[j].converged
        else:
            assert st[j].converged and st[j].iterations == ref[j].iterations
            assert torch.equal(X[:, j], Y[:, j])
    Bt[7, columns] = 0.0
    s.solve_multi(Bt, Y, K)   # the solver is as before
    assert torch.equal(X, Y)
