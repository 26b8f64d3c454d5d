"""Products of values up to the largest finite ones: the element transforms add up to eight staged
values before any scaling, which may not overflow where the product itself does not.

Scaling x by a power of two scales every term and its fixed-point grid alike, so the product of
2^k x is 2^k times that of x to the bit, up to the largest k for which x stays finite (the factors
2^-8 keep the results finite too).  Oracle comparisons of the products at ordinary sizes are
elsewhere; no tolerance here but equality.
"""
import numpy as np
import pytest

import dendro_amd as da
from tests.meshes import hierarchy

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

DT = {da.F64: torch.float64, da.F32: torch.float32}
TOP = {da.F64: 1024, da.F32: 128}   # |x| < 1 scaled by 2^TOP is still finite
SMALL = 2.0 ** -8


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    da.init(0)
    return torch.device("cuda:0")


def times2(t, k):
    """t 2^k, in steps that are themselves finite"""
    for s in (k // 2, k - k // 2):
        t = t * 2.0 ** s
    return t


def mesh(L, coef):
    rng = np.random.default_rng(8)
    kap = SMALL * 10.0 ** rng.uniform(-1, 0, L.n_elem) if coef != "uniform" else None
    mas = SMALL * rng.uniform(0.5, 1, L.n_elem) if coef == "kappa_mass" else None
    m = da.Mesh(L)
    m.set_coefficients(kap, mas, SMALL, SMALL)
    return m


@pytest.fixture(scope="module")
def hier():
    return hierarchy("clusters", 9000, 10, 1, seed=6, min_coarse=1)


@pytest.mark.parametrize("coef", ["uniform", "kappa", "kappa_mass"])
@pytest.mark.parametrize("prec", [da.F64, da.F32])
def test_product(dev, hier, coef, prec):
    L = hier.fine
    m = mesh(L, coef)
    m.set_boundary(hier.damg.boundary(0))
    x = torch.tensor(np.random.default_rng(9).uniform(0.5, 0.999, L.n_node), dtype=DT[prec], device=dev)
    for call in (m.matvec, m.matvec_dirichlet):
        for block in (256, 512, 1024):
            m.set_tile(256, block)
            y, big = torch.empty_like(x), torch.empty_like(x)
            call(x, y, prec=prec)
            for k in (TOP[prec] - 5, TOP[prec] - 3, TOP[prec] - 2, TOP[prec]):
                call(times2(x, k), big, prec=prec)
                assert torch.equal(big, times2(y, k)), (call.__name__, block, k)
    x[L.n_node // 2] = float("inf")
    m.matvec(x, y, prec=prec)
    assert torch.isnan(y[L.n_node // 2])


@pytest.mark.parametrize("coef", ["uniform", "kappa", "kappa_mass"])
@pytest.mark.parametrize("prec", [da.F64, da.F32])
def test_batched_product(dev, hier, coef, prec):
    """Columns of very different sizes in one slice: each is the column alone, scaled."""
    L, k = hier.fine, 16
    m = mesh(L, coef)
    x = torch.tensor(np.random.default_rng(9).uniform(0.5, 0.999, (L.n_node, k)), dtype=DT[prec], device=dev)
    top = TOP[prec]
    e = [(0, top, top - 1, -60, top - 3, 3, top - 2, -20)[j % 8] for j in range(k)]
    big = torch.stack([times2(x[:, j], e[j]) for j in range(k)], 1).contiguous()
    for variant in (0, 2, 3, 4, 5, 6) if prec == da.F32 else (6,):
        m.set_tile_multi(256, variant)
        y, z = torch.empty_like(x), torch.empty_like(x)
        m.matvec_multi(x, y, k, prec=prec)
        m.matvec_multi(big, z, k, prec=prec)
        for j in range(k):
            assert torch.equal(z[:, j], times2(y[:, j], e[j])), (variant, j, e[j])


@pytest.mark.parametrize("mu,lam,top", [(SMALL, SMALL, 1024), (2.0 ** 500, 2.0 ** 500, 516)])
def test_elasticity_product(dev, hier, mu, lam, top):
    """top: the largest x for which the results stay finite"""
    L = hier.fine
    m = da.Mesh(L)
    m.set_elasticity(mu, lam)
    x = torch.tensor(np.random.default_rng(9).uniform(0.5, 0.999, (L.n_node, 3)), device=dev)
    y, big = torch.empty_like(x), torch.empty_like(x)
    m.matvec_elasticity(x, y)
    for k in (top - 5, top - 3, top):
        m.matvec_elasticity(times2(x, k), big)
        assert torch.equal(big, times2(y, k)), k


@pytest.mark.parametrize("npts,levels", [(2000, 2), (32000, 5)])
@pytest.mark.parametrize("prec", [da.F64, da.F32])
def test_vcycle(dev, npts, levels, prec):
    """Sweeps and residuals, two per launch (small levels) and single: the iterates of a positive
    right-hand side reach the largest values, sums over the coarse rows stay far below."""
    h = hierarchy("clusters", npts, 10, levels, seed=4, min_coarse=50)
    assert h.fine.n_elem > 60000 if levels > 2 else h.fine.n_elem < 20000
    ms = [da.Mesh(L) for L in h.levels]
    for m in ms:
        m.set_coefficients(None, None, 1.0, 1.0)
    ts = [da.Transfer(ms[l - 1], ms[l], *h.transfers[l - 1]) for l in range(1, h.n)]
    r = torch.tensor(np.random.default_rng(5).uniform(0.5, 1, h.fine.n_node), device=dev)
    r = r.float().double()
    for pre, post in ((2, 2), (3, 1)):
        s = da.Solver(ms, ts, da.default_params(omega=2.0 / 3.0, nu_pre=pre, nu_post=post, vcycle_prec=prec))
        z, big = torch.empty_like(r), torch.empty_like(r)
        s.vcycle(r, z)
        k = TOP[prec] - 2 - int(np.ceil(np.log2(float(z.abs().max()))))
        s.vcycle(times2(r, k), big)
        assert torch.isfinite(big).all()
        assert torch.equal(big, times2(z, k)), (pre, post)
