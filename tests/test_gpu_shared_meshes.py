"""Solvers that share meshes: creating one only reads them, so another may run on its own thread
meanwhile, and each follows new coefficients by itself.  Equal bits throughout: the same kernels on the
same tiles.
"""
import threading

import numpy as np
import pytest

import dendro_amd as da
from tests.meshes import hierarchy, var_coefficients

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def shared():
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    da.init(0)
    h = hierarchy("clusters", 2000, 10, 3, seed=4, min_coarse=50)
    assert 2000 < h.fine.n_elem < 20000   # a size smoothed two sweeps per launch in both precisions
    c = var_coefficients(h, mass_base=1.0)
    return h, c


def meshes(h, c, scale=1.0):
    ms = [da.Mesh(L) for L in h.levels]
    for m, (k, q) in zip(ms, c):
        m.set_coefficients(k * scale, q * scale)
    return ms, [da.Transfer(ms[l - 1], ms[l], *h.transfers[l - 1]) for l in range(1, h.n)]


def solver(ms, ts, prec, **kw):
    return da.Solver(ms, ts, da.default_params(omega=2.0 / 3.0, nu_pre=2, nu_post=2, rtol=1e-8, max_it=40,
                                               norm_type=da.NORM_UNPRECONDITIONED, vcycle_prec=prec, **kw))


@pytest.mark.parametrize("prec", [da.F64, da.F32])
def test_each_solver_follows_new_coefficients(shared, prec):
    h, c = shared
    ms, ts = meshes(h, c)
    a, b = solver(ms, ts, prec, use_graph=1), solver(ms, ts, prec)
    r = torch.tensor(np.random.default_rng(3).uniform(-1, 1, h.fine.n_node), device="cuda:0")
    x, y = torch.empty_like(r), torch.empty_like(r)
    a.solve(r, x)
    b.vcycle(r, x)
    for m, (k, q) in zip(ms, c):
        m.set_coefficients(k * 3.0, q * 3.0)
    ref = solver(*meshes(h, c, 3.0), prec)
    for s in (a, b):
        s.vcycle(r, x)
        ref.vcycle(r, y)
        assert torch.equal(x, y)
        s.solve(r, x)
        ref.solve(r, y)
        assert torch.equal(x, y)


def test_creation_beside_a_running_solver(shared):
    h, c = shared
    ms, ts = meshes(h, c)
    s = solver(ms, ts, da.F64)   # its coarse inverse sets up the library's handles
    r = torch.tensor(np.random.default_rng(3).uniform(-1, 1, h.fine.n_node), device="cuda:0")
    x = torch.empty_like(r)
    st0, _ = s.solve(r, x)
    ref = x.clone()
    torch.cuda.synchronize()
    wrong, stop = [], threading.Event()

    def run():
        y = torch.empty_like(r)
        while not stop.is_set():
            st, _ = s.solve(r, y)   # returns when x is complete
            if st.iterations != st0.iterations or not torch.equal(y, ref):
                wrong.append(st.iterations)

    t = threading.Thread(target=run)
    t.start()
    try:
        for _ in range(6):
            for prec in (da.F32, da.F64):
                other = solver(ms, ts, prec)
                z = torch.empty_like(r)
                other.solve(r, z)
                del other
    finally:
        stop.set()
        t.join()
    assert not wrong
