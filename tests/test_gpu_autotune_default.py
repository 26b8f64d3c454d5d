"""The autotuners time the default tiling among their candidates, so a tuned mesh is not slower than an
untouched one.  Bar: 15% (the shortest of nine batches repeats within 5%; the nearest listed tile size of
the batched product costs 25% and more on these meshes).
"""
import pytest

import dendro_amd as da
from tests.meshes import hierarchy

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

BAR = 1.15


def shortest(f, n=100):
    for _ in range(20):
        f()
    ts = []
    for _ in range(9):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(n):
            f()
        b.record()
        b.synchronize()
        ts.append(a.elapsed_time(b) / n * 1e3)
    return min(ts)


@pytest.mark.parametrize("npts,depth", [(300, 5), (900, 6)])
def test_tuned_is_not_slower(npts, depth):
    da.init(0)
    L = hierarchy("gauss", npts, depth, 1, min_coarse=1).fine
    m = da.Mesh(L)
    m.set_coefficients(None, None)
    k = 8
    x = torch.rand(L.n_node, k, dtype=torch.float32, device="cuda:0")
    y = torch.empty_like(x)
    before = shortest(lambda: m.matvec_multi(x, y, k, prec=da.F32))
    r = m.autotune_multi(k)
    after = shortest(lambda: m.matvec_multi(x, y, k, prec=da.F32))
    print(L.n_elem, r, f"{before:.2f} -> {after:.2f} us")
    assert after <= BAR * before
    x = torch.rand(L.n_node, dtype=torch.float64, device="cuda:0")
    y = torch.empty_like(x)
    before = shortest(lambda: m.matvec(x, y))
    r = m.autotune()
    after = shortest(lambda: m.matvec(x, y))
    print(L.n_elem, r, f"{before:.2f} -> {after:.2f} us")
    assert after <= BAR * before
