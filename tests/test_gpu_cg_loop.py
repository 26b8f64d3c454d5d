"""The CG loop on the GPU, whose stopping test runs on the device while the host queues an
iteration ahead: iteration counts, norms and solutions against the oracle's PCG for both norms,
loose and tight tolerances, iteration limits, a zero right-hand side and tilings with more
partials of p.w than one workgroup sums.

The solver and the oracle run the same FP64 recurrences, differing by rounding: with at most 12
iterations each reducing the residual by 5 or more, the norms agree to 1e-9 of the initial one and
the solutions to 1e-8 (the error bound of a residual reduced by 1e-8 or of equal iterates).
"""
import numpy as np
import pytest

import dendro_amd as da
import oracle
from tests.meshes import hierarchy, rel_err, var_coefficients

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def problem():
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    da.init(0)
    h = hierarchy("clusters", 6000, 10, 3, seed=4, min_coarse=50)
    coefs = var_coefficients(h, mass_base=1.0)
    mg = oracle.MG([(h.levels[l], coefs[l][0], coefs[l][1], 1.0, 1.0) for l in range(h.n)], omega=2.0 / 3.0, nu_pre=2,
                   nu_post=2)
    b = np.random.default_rng(17).uniform(-1, 1, h.fine.n_node)
    return h, coefs, mg, b


def _solve(problem, b, tile=None, **kw):
    h, coefs, _, _ = problem
    ms = []
    for l in range(h.n):
        m = da.Mesh(h.levels[l])
        m.set_coefficients(*coefs[l])
        ms.append(m)
    if tile:
        ms[-1].set_tile(*tile)
    ts = [da.Transfer(ms[l - 1], ms[l], *h.transfers[l - 1]) for l in range(1, h.n)]
    s = da.Solver(ms, ts, da.default_params(omega=2.0 / 3.0, nu_pre=2, nu_post=2, **kw))
    bt = torch.tensor(b, dtype=torch.float64, device="cuda:0")
    out = []
    for _ in range(2):   # the second solve starts from the first one's leftovers
        x = torch.full_like(bt, float("nan"))
        st, hist = s.solve(bt, x, history_len=64)
        out.append((st, np.array(hist), x.cpu().numpy()))
    assert out[0][0].iterations == out[1][0].iterations
    assert np.array_equal(out[0][2], out[1][2])
    return out[0] + (ms[-1].tile_info(),)


@pytest.mark.parametrize("norm", [da.NORM_UNPRECONDITIONED, da.NORM_PRECONDITIONED])
@pytest.mark.parametrize("rtol,max_it", [(1e-8, 100), (0.3, 100), (1e-3, 100), (1e-8, 1), (1e-8, 2), (1e-8, 3)])
def test_loop_matches_oracle(problem, norm, rtol, max_it):
    _, _, mg, b = problem
    xo, its, conv, ho = mg.pcg(b, rtol=rtol, max_it=max_it, norm_type=norm)
    for graph in (0, 1):
        st, hist, x, _ = _solve(problem, b, rtol=rtol, max_it=max_it, norm_type=norm, use_graph=graph)
        assert st.iterations == its and bool(st.converged) == bool(conv)
        n = its + 1
        assert np.max(np.abs(hist[:n] - np.array(ho)[:n])) <= 1e-9 * ho[0]
        assert rel_err(x, xo) <= 1e-8


@pytest.mark.parametrize("prec", [da.F64, da.F32])
@pytest.mark.parametrize("norm", [da.NORM_UNPRECONDITIONED, da.NORM_PRECONDITIONED])
def test_zero_rhs_and_no_iterations(problem, norm, prec):
    b = problem[3]
    st, _, x, _ = _solve(problem, np.zeros_like(b), rtol=1e-8, max_it=50, norm_type=norm, vcycle_prec=prec, use_graph=1)
    assert st.iterations == 0 and st.converged and not x.any()
    st, _, x, _ = _solve(problem, b, rtol=1e-8, max_it=0, norm_type=norm, vcycle_prec=prec)
    assert st.iterations == 0 and not st.converged and not x.any()


def test_many_and_few_partials(problem):
    """2300 tiles (their partials of p.w are summed by a kernel of their own) and 30, against the
    default tiling."""
    h = hierarchy("clusters", 32000, 10, 5, seed=4, min_coarse=50)
    b = np.random.default_rng(18).uniform(-1, 1, h.fine.n_node)
    prob = (h, var_coefficients(h, mass_base=1.0), None, b)
    kw = dict(rtol=1e-8, max_it=100, norm_type=da.NORM_UNPRECONDITIONED, use_graph=1)
    ref = _solve(prob, b, **kw)
    tiles = []
    for tile in ((64, 512), (8192, 1024)):
        st, _, x, info = _solve(prob, b, tile=tile, **kw)
        tiles.append(info["n_tiles"])
        assert st.iterations == ref[0].iterations and rel_err(x, ref[2]) <= 1e-8
    assert tiles[0] > 2048 > 512 > tiles[1]


@pytest.mark.parametrize("k", [8, 24])
@pytest.mark.parametrize("norm", [da.NORM_UNPRECONDITIONED, da.NORM_PRECONDITIONED])
@pytest.mark.parametrize("rtol,max_it", [(1e-8, 100), (0.3, 100), (1e-8, 2), (1e-8, 0)])
def test_batched_loop(problem, norm, rtol, max_it, k):
    """Columns of different difficulty (smooth, rough, zero) against single solves with the same FP32
    V-cycle: equal iterations, and solutions that agree to what their residuals leave open."""
    h, coefs, _, b = problem
    ms = []
    for l in range(h.n):
        m = da.Mesh(h.levels[l])
        m.set_coefficients(*coefs[l])
        ms.append(m)
    ts = [da.Transfer(ms[l - 1], ms[l], *h.transfers[l - 1]) for l in range(1, h.n)]
    rng = np.random.default_rng(19)
    B = rng.uniform(-1, 1, (h.fine.n_node, k))
    B[:, 1] = 1.0
    B[:, 3] = 0.0
    for graph in (0, 1):
        s = da.Solver(ms, ts, da.default_params(omega=2.0 / 3.0, nu_pre=2, nu_post=2, rtol=rtol, max_it=max_it,
                                                norm_type=norm, use_graph=graph, vcycle_prec=da.F32))
        Bt = torch.tensor(B, dtype=torch.float64, device="cuda:0")
        X, Y = torch.full_like(Bt, float("nan")), torch.empty_like(Bt)
        st = s.solve_multi(Bt, X, k)
        s.solve_multi(Bt, Y, k)
        assert torch.equal(X, Y)
        assert st[3].iterations == 0 and st[3].converged and not X[:, 3].any()
        for j in (0, 1, k - 1):
            bt, x = Bt[:, j].contiguous(), torch.empty_like(Bt[:, 0])
            one, _ = s.solve(bt, x)
            assert st[j].iterations == one.iterations and st[j].converged == one.converged
            if max_it:
                assert rel_err(X[:, j].cpu().numpy(), x.cpu().numpy()) <= max(1e-4, 10 * rtol if rtol < 0.1 else 0.0)
