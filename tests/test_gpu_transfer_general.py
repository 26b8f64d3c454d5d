"""The general transfer kernels, which run where a block of rows has more distinct columns than the LDS
forms take (2047).  Node numbers that follow the octree's order never come near; here the nodes are
renumbered so that the first rows share no column: 256 fine nodes at the centres of coarse elements
without a common vertex (2048 columns), 128 coarse nodes with 27 fine nodes around each.  With and
without boundary flags, both precisions, against the oracle in the octree's numbering.

Tolerances: each result is a sum of at most 64 products with weights that are exact in FP32, so
64 2^-53 and 64 2^-24 of the sum of absolute terms, a few times the result's norm: 1e-13 and 1e-5.
"""
import numpy as np
import pytest

import dendro_amd as da
import oracle
from tests.meshes import hierarchy, rel_err

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

LIMIT = 2047   # columns of a block the LDS forms take


class Renumbered:
    """A level whose node n is called new[n]."""

    def __init__(self, L, new):
        self.__dict__.update(L.__dict__)
        self.nlist = np.ascontiguousarray(new[L.nlist].astype(np.uint32))


def first(n, chosen):
    """new numbers that put the chosen nodes first and keep the order of the others"""
    rest = np.ones(n, bool)
    rest[chosen] = False
    new = np.empty(n, np.int64)
    new[np.concatenate([chosen, np.nonzero(rest)[0]])] = np.arange(n)
    return new


def disjoint(rows, columns, count):
    """the first `count` rows (in a random order) whose columns no earlier one has"""
    used, out = set(), []
    for i in np.random.default_rng(1).permutation(rows):
        c = columns(i)
        if used.isdisjoint(c):
            used.update(c)
            out.append(i)
            if len(out) == count:
                break
    assert len(out) == count
    return np.array(out), len(used)


def test_general_kernels():
    da.init(0)
    h = hierarchy("lognormal", 250000, 11, 2, seed=3, min_coarse=1)
    C, F = h.levels
    celem, pos = h.transfers[0]
    assert C.n_node >= 80000   # the restriction's blocks of 128 rows
    # entries through coarse elements without hanging vertices: vertex k has a weight at a node on
    # or opposite none of its sides
    plain = C.hnmask[celem] == 0
    t = np.stack([pos % 3, pos // 3 % 3, pos // 9], 1)
    centre = np.nonzero(plain & (t == 1).all(1))[0]
    fine, n_cols = disjoint(centre, lambda j: C.nlist[celem[j]].tolist(), 256)
    assert n_cols > LIMIT
    rows = {}
    for k in range(8):
        bits = np.array([k & 1, k >> 1 & 1, k >> 2 & 1])
        has = plain & ((t == 1) | (t == 2 * bits)).all(1)
        for j in np.nonzero(has)[0]:
            rows.setdefault(int(C.nlist[celem[j], k]), []).append(int(j))
    full = [i for i, r in rows.items() if len(r) == 27]
    coarse, n_cols = disjoint(full, lambda i: rows[i], 128)
    assert n_cols > LIMIT
    cn, fn = first(C.n_node, coarse), first(F.n_node, fine)
    ms = [da.Mesh(Renumbered(C, cn)), da.Mesh(Renumbered(F, fn))]
    ce, po = np.empty_like(celem), np.empty_like(pos)
    ce[fn], po[fn] = celem, pos
    tr = da.Transfer(ms[0], ms[1], ce, po)
    rng = np.random.default_rng(9)
    f, c, x = rng.uniform(-1, 1, F.n_node), rng.uniform(-1, 1, C.n_node), rng.uniform(-1, 1, F.n_node)
    f, c, x = (v.astype(np.float32).astype(np.float64) for v in (f, c, x))
    bc, bf = h.damg.boundary(0), h.damg.boundary(1)
    for dirichlet in (False, True):
        keep_c, keep_f = (bc == 0, bf == 0) if dirichlet else (np.ones(C.n_node, bool), np.ones(F.n_node, bool))
        for m, b, new in ((ms[0], bc, cn), (ms[1], bf, fn)):
            flags = np.empty_like(b)
            flags[new] = b
            m.set_boundary(flags if dirichlet else None)
        rc = keep_c * oracle.restrict(C, F, f * keep_f)
        pc = keep_f * oracle.prolong(C, F, c * keep_c)
        for prec, dt, tol in ((da.F64, torch.float64, 1e-13), (da.F32, torch.float32, 1e-5)):
            def up(a, new):
                b = np.empty_like(a)
                b[new] = a
                return torch.tensor(b, dtype=dt, device="cuda:0")
            ft, ct, xt = up(f, fn), up(c, cn), up(x, fn)
            out = torch.empty_like(ct)
            tr.restrict(ft, out, prec=prec)
            assert rel_err(out.double().cpu().numpy()[cn], rc) <= tol
            y = torch.empty_like(xt)
            tr.prolong_add(ct, xt, y, prec=prec)
            assert rel_err(y.double().cpu().numpy()[fn], x + pc) <= tol
            tr.prolong_add(ct, None, y, prec=prec)
            assert rel_err(y.double().cpu().numpy()[fn], pc) <= tol
