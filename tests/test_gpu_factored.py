"""The factored element product (the operator kernels' default) on the GPU: against the oracle and
against the per-type stencil rows at tile sizes and meshes whose tiles end in partial
wavefronts, for every coefficient form, block size and precision.

Tolerances: an FP64 term is rounded to 2^-50 of its tile's bound, so 1e-12 relative (the bar of
every FP64 product here); an FP32 term to 2^-24 of it or finer per contribution, with at most 32
contributions to a node and a bound a few times the largest row, so 5e-6.
"""
import numpy as np
import pytest

import dendro_amd as da
import oracle
from tests.meshes import hierarchy

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    da.init(0)
    return torch.device("cuda:0")


MESHES = {"one": ("uniform", 1, 3), "few": ("clusters", 9, 6), "edge": ("lognormal", 700, 8), "mid": ("clusters", 9000, 10)}


@pytest.mark.parametrize("coef", ["helmholtz", "laplacian", "kappa", "kappa_mass"])
@pytest.mark.parametrize("mesh", sorted(MESHES))
def test_factored_product(dev, mesh, coef):
    L = hierarchy(*MESHES[mesh], 1, seed=6, min_coarse=1).fine
    rng = np.random.default_rng(8)
    x = rng.uniform(-1, 1, L.n_node)
    kap = 10.0 ** rng.uniform(-1, 1, L.n_elem) if coef.startswith("kappa") else None
    mas = rng.uniform(0.5, 2, L.n_elem) if coef == "kappa_mass" else None
    mf = 0.0 if coef == "laplacian" else 1.0
    ref = oracle.matvec(L, x, kappa=kap, mass=mas, lap_fac=1.0, mass_fac=mf)
    # each node's scale: the 2-norm of A x can be tiny against its terms (a one-element mesh)
    size = np.linalg.norm(oracle.diagonal(L, kappa=kap, mass=mas, lap_fac=1.0, mass_fac=mf) * np.abs(x))
    m = da.Mesh(L)
    m.set_coefficients(kap, mas, 1.0, mf)
    for tile, block in ((64, 256), (65, 512), (1000, 256), (1000, 1024)):
        for prec, dt, tol in ((da.F64, torch.float64, 1e-12), (da.F32, torch.float32, 5e-6)):
            m.set_tile(tile, block)
            xt = torch.tensor(x, dtype=dt, device=dev)
            y, yr = torch.empty_like(xt), torch.empty_like(xt)
            m.matvec(xt, y, prec=prec)
            y8 = torch.empty_like(xt)
            m.matvec(xt * 8, y8, prec=prec)
            r = da.Mesh(L)
            r.set_coefficients(kap, mas, 1.0, mf)
            r.set_tile(tile, block)
            r.set_lane_stencils(da.ROWS_TYPE)
            r.matvec(xt, yr, prec=prec)
            err = np.linalg.norm(y.cpu().numpy() - ref) / size
            print(f"{mesh} {coef} tile {tile} block {block} prec {prec}: {err:.2e}")
            assert err <= tol
            assert np.linalg.norm((y - yr).double().cpu().numpy()) / size <= tol
            assert torch.equal(y8, y * 8)   # the scale of x passes through exactly
    xt[L.n_node // 2] = float("inf")
    m.matvec(xt, y, prec=da.F32)
    assert torch.isnan(y[L.n_node // 2])


@pytest.mark.parametrize("dirichlet", [False, True])
@pytest.mark.parametrize("mesh", sorted(MESHES))
def test_factored_elasticity(dev, mesh, dirichlet):
    h = hierarchy(*MESHES[mesh], 1, seed=6, min_coarse=1)
    L = h.fine
    bdy = h.damg.boundary(0) if dirichlet else None
    x = np.random.default_rng(9).uniform(-1, 1, (L.n_node, 3))
    m = da.Mesh(L)
    m.set_boundary(bdy)
    xt = torch.tensor(x, device=dev)
    y = torch.empty_like(xt)
    for mu, lam in ((1.0, 1.5), (0.7, -0.3)):
        m.set_elasticity(mu, lam)
        m.matvec_elasticity(xt, y)
        ref = oracle.matvec_elasticity(L, x, mu, lam, bdy).reshape(-1, 3)
        got = y.cpu().numpy()
        err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
        print(f"{mesh} mu {mu} lambda {lam}: {err:.2e}")
        assert err <= 1e-12
        if dirichlet:
            assert np.array_equal(got[bdy != 0], x[bdy != 0])


@pytest.mark.parametrize("fn", [dict(kind=da.FN_COS_SUM, nfreq=1), dict(kind=da.FN_COS_SUM, nfreq=19, a0=1.0, a1=0.5),
                                dict(kind=da.FN_GAUSSIANS), dict(kind=da.FN_POLY, poly=[1, -2, .5, 3, .25, -1, 2, -.75])])
@pytest.mark.parametrize("mesh", sorted(MESHES) + ["shuffled"])
def test_quadrature(dev, mesh, fn):
    """Load vector and L2 error on meshes of one to many workgroups (partial ones among them), with
    one and several passes over the frequencies; shuffled: elements in random order, so that a
    workgroup holds more coordinate intervals than its table takes at once."""
    L = hierarchy(*MESHES["mid" if mesh == "shuffled" else mesh], 1, seed=6, min_coarse=1).fine
    if mesh == "shuffled":
        o = np.random.default_rng(3).permutation(L.n_elem)
        for name in ("nlist", "child", "hnmask", "lev", "anchor"):
            setattr(L, name, np.ascontiguousarray(getattr(L, name)[o]))
    m = da.Mesh(L)
    m.set_geometry(L.anchor)
    f = da.function(**fn)
    b = torch.empty(L.n_node, dtype=torch.float64, device=dev)
    m.rhs_quadrature(f, b)
    ref = oracle.rhs_quadrature(L, **fn)
    got = b.cpu().numpy()
    # terms of size sum |w f phi|: one is at most the function's maximum times the mass row
    size = np.linalg.norm(ref) + 1e-3 * np.linalg.norm(oracle.rhs_quadrature(L, kind=da.FN_POLY, poly=[1] + [0] * 7))
    assert np.linalg.norm(got - ref) <= 1e-12 * size
    u = np.random.default_rng(4).uniform(-1, 1, L.n_node)
    e = m.l2_error(f, torch.tensor(u, device=dev))
    e_ref = oracle.l2_error(L, u, **fn)
    assert abs(e - e_ref) <= 1e-12 * e_ref
    assert e == m.l2_error(f, torch.tensor(u, device=dev))   # summed in a fixed order
