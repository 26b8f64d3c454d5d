"""The workloads whose time is followed: single operators, transfers and whole solves on seeded octrees.

A case names its octree; coefficients and vectors come from the seed.  prepare() keeps what a
program that solves on this mesh keeps (device meshes, transfers, a solver) and run() makes one
pass through the public calls of dendro_amd.  Tilings are the library's defaults, as the C++ facade and its
driver leave them.  exact() evaluates the same quantities in 64 bits with plain torch: the
mesh arrays (node lists, child numbers, hanging masks, levels, transfer maps) are inputs; the
element matrices, hanging-node constraints and interpolation weights are formed here from the
trilinear shape functions.
"""
import functools

import numpy as np
import torch

import dendro_amd as da

KINDS = {"gauss": da.PTS_GAUSS, "lognormal": da.PTS_LOGNORMAL, "mixed": da.PTS_MIXED,
         "clusters": da.PTS_CLUSTERS, "uniform": da.PTS_UNIFORM}
DTYPE = {"f64": torch.float64, "f32": torch.float32}
PREC = {"f64": da.F64, "f32": da.F32}
OMEGA = 2.0 / 3.0

LISTED = [
    # the smallest product a program makes: a mesh of a few thousand elements, where the launch counts
    {"name": "matvec_small", "op": "matvec", "points": "gauss", "n": 3000, "depth": 6, "coef": "helmholtz",
     "prec": "f64"},
    # the FP64 product of a Helmholtz problem of ordinary size (100k Gaussian points)
    {"name": "matvec_gauss", "op": "matvec", "points": "gauss", "n": 100000, "depth": 8, "coef": "helmholtz",
     "prec": "f64"},
    # the FP64 product with an element coefficient (1M log-normal points, the Poisson workload)
    {"name": "matvec_kappa", "op": "matvec", "points": "lognormal", "n": 1000000, "depth": 12, "coef": "kappa",
     "prec": "f64"},
    # a large mesh: half uniform, half clustered points, where memory counts
    {"name": "matvec_large", "op": "matvec", "points": "mixed", "n": 2000000, "depth": 13, "coef": "helmholtz",
     "prec": "f64"},
    # the product of a Dirichlet problem (boundary rows and columns masked)
    {"name": "dirichlet", "op": "dirichlet", "points": "lognormal", "n": 300000, "depth": 11, "coef": "helmholtz",
     "prec": "f64"},
    # both grid transfers of a V-cycle in its working precision: residual down, correction up
    {"name": "transfer", "op": "transfer", "points": "lognormal", "n": 300000, "depth": 11, "prec": "f32"},
    # 32 right-hand sides at once: the batched V-cycle's operator
    {"name": "multi", "op": "multi", "points": "lognormal", "n": 300000, "depth": 11, "coef": "kappa",
     "prec": "f32", "k": 32},
    # linear elasticity, three unknowns per node
    {"name": "elasticity", "op": "elasticity", "points": "gauss", "n": 100000, "depth": 8},
    # load vector of an analytic source and the L2 error of a nodal solution
    {"name": "source_and_error", "op": "fem", "points": "gauss", "n": 100000, "depth": 8, "fn": "cos", "nfreq": 9},
    # one FP64 multigrid V-cycle (a program's own Krylov loop calls it), coefficients with contrast and mass
    {"name": "vcycle", "op": "vcycle", "points": "clusters", "n": 60000, "depth": 10, "coef": "kappa_mass",
     "levels": 5},
    # the whole solve to 1e-8: FP32 V-cycle inside FP64 CG, pure Neumann problem
    {"name": "solve", "op": "solve", "points": "lognormal", "n": 300000, "depth": 11, "coef": "kappa",
     "prec": "f32", "levels": 5},
    # a batch of solves on one mesh
    {"name": "solve_batch", "op": "solve_multi", "points": "gauss", "n": 30000, "depth": 8, "coef": "helmholtz",
     "levels": 4, "k": 16},
]

# points per case of a kind of work: the listed ones lie inside these ranges
RANGES = {"matvec": (500, 300000), "dirichlet": (500, 300000), "transfer": (2000, 300000), "multi": (1000, 200000),
          "elasticity": (500, 100000), "fem": (500, 100000), "vcycle": (3000, 60000), "solve": (3000, 200000),
          "solve_multi": (2000, 20000)}


def listed():
    return [dict(c) for c in LISTED]


def draw(rng):
    op = rng.choice(sorted(RANGES))
    lo, hi = RANGES[op]
    n = int(lo * (hi / lo) ** rng.random())
    points = rng.choice(sorted(KINDS))
    # depth: enough levels for the points' density, and up to three more for the clustered ones
    depth = max(4, int(round(np.log2(n) / 3.0)) + rng.randint(1, 4))
    c = {"op": op, "points": points, "n": n, "depth": min(depth, 14)}
    if op in ("matvec", "dirichlet", "transfer", "multi"):
        c["prec"] = rng.choice(["f64", "f32"])
    if op in ("matvec", "dirichlet", "multi", "vcycle", "solve", "solve_multi"):
        c["coef"] = rng.choice(["helmholtz", "kappa", "kappa_mass"])
    if op in ("vcycle", "solve", "solve_multi"):
        c["levels"] = rng.choice([4, 5, 6])
    if op == "vcycle" and c["coef"] == "kappa":
        c["coef"] = "kappa_mass"
    if op == "solve":
        c["prec"] = rng.choice(["f64", "f32"])
    if op in ("multi", "solve_multi"):
        c["k"] = rng.choice([8, 16, 24, 32])
    if op == "fem":
        c["fn"] = rng.choice(["cos", "gaussians", "poly"])
        c["nfreq"] = rng.randint(1, 9)
    return c


# ---------------------------------------------------------------- inputs
@functools.lru_cache(maxsize=2)
def _octree_hierarchy(points, n, depth, levels):
    pts = da.points(KINDS[points], n, 5, 31)
    return da.DAMG(da.Octree.from_points(pts, depth), levels, 500)


def _hierarchy(case):
    """The host mesh of a case (octree, DA hierarchy); a program builds or loads it once."""
    levels = case.get("levels", 2 if case["op"] == "transfer" else 1)
    return _octree_hierarchy(case["points"], case["n"], case["depth"], levels)


def _coefficients(case, damg, seed):
    """Per level (kappa, mass) or (None, None): kappa_e = 10^U(-1, 1), mass_e = U(0.5, 2) on the finest
    level, averaged to the coarser ones."""
    coef = case.get("coef", "helmholtz")
    if coef == "helmholtz":
        return [(None, None)] * damg.nlevels
    rng = np.random.default_rng([seed, 1])
    ne = damg.info(damg.nlevels - 1).n_elem
    kf = 10.0 ** rng.uniform(-1, 1, ne)
    mf = rng.uniform(0.5, 2.0, ne) if coef == "kappa_mass" else None
    return [damg.coarsen_coefficients(kf, mf, l) for l in range(damg.nlevels)]


def _uniform(seed, shape, dtype):
    g = torch.Generator(device="cuda")
    g.manual_seed(7919 * seed + 17)
    return torch.rand(shape, generator=g, device="cuda", dtype=dtype) * 2 - 1


def _function(case):
    if case["fn"] == "cos":
        return da.function(da.FN_COS_SUM, nfreq=case["nfreq"], a0=1.0, a1=1.0)
    if case["fn"] == "gaussians":
        return da.function(da.FN_GAUSSIANS)
    return da.function(da.FN_POLY, poly=[0.3, 1.0, -0.7, 0.4, 0.9, -1.1, 0.6, 0.2])


def _null_space(case):
    return int(case.get("coef") == "kappa")   # no mass term: constants are in the kernel


def prepare(case, seed):
    da.init(0)
    op = case["op"]
    damg = _hierarchy(case)
    coefs = _coefficients(case, damg, seed)
    first = 0 if op in ("transfer", "vcycle", "solve", "solve_multi") else damg.nlevels - 1
    meshes = []
    for l in range(first, damg.nlevels):
        m = da.Mesh(damg.level(l))
        m.set_coefficients(*coefs[l], 1.0, 1.0)
        meshes.append(m)
    fine = meshes[-1]
    n = fine.n_node
    s = {"case": case, "mesh": fine, "meshes": meshes}
    if op == "matvec":
        s["x"] = _uniform(seed, n, DTYPE[case["prec"]])
        s["y"] = torch.empty_like(s["x"])
    elif op == "dirichlet":
        fine.set_boundary(damg.boundary(damg.nlevels - 1))
        s["x"] = _uniform(seed, n, DTYPE[case["prec"]])
        s["y"] = torch.empty_like(s["x"])
    elif op == "multi":
        s["x"] = _uniform(seed, (n, case["k"]), DTYPE[case["prec"]])
        s["y"] = torch.empty_like(s["x"])
    elif op == "elasticity":
        fine.set_elasticity(1.0, 1.5)
        s["x"] = _uniform(seed, (n, 3), torch.float64)
        s["y"] = torch.empty_like(s["x"])
    elif op == "fem":
        fine.set_geometry(damg.level(damg.nlevels - 1).anchor)
        s["f"] = _function(case)
        s["u"] = _uniform(seed, n, torch.float64)
        s["b"] = torch.empty_like(s["u"])
    else:
        s["transfers"] = [da.Transfer(meshes[l - 1], meshes[l], *damg.transfer(l)) for l in range(1, len(meshes))]
    if op == "transfer":
        dt = DTYPE[case["prec"]]
        s["r"] = _uniform(seed, n, dt)
        s["c"] = torch.empty(meshes[0].n_node, dtype=dt, device="cuda")
        s["e"] = _uniform(seed + 1, meshes[0].n_node, dt)
        s["x"] = _uniform(seed + 2, n, dt)
        s["y"] = torch.empty_like(s["x"])
    elif op in ("vcycle", "solve", "solve_multi"):
        p = da.default_params(omega=OMEGA, nu_pre=2, nu_post=2, max_it=200, rtol=1e-8, use_graph=1,
                              norm_type=da.NORM_UNPRECONDITIONED, null_space=_null_space(case),
                              vcycle_prec=PREC[case.get("prec", "f64")])
        s["solver"] = da.Solver(meshes, s["transfers"], p)
        shape = (n, case["k"]) if op == "solve_multi" else n
        s["b"] = _uniform(seed, shape, torch.float64)
        s["x"] = torch.empty_like(s["b"])
    return s


def run(s):
    case = s["case"]
    op, m = case["op"], s["mesh"]
    if op == "matvec":
        m.matvec(s["x"], s["y"], PREC[case["prec"]])
        return s["y"]
    if op == "dirichlet":
        m.matvec_dirichlet(s["x"], s["y"], PREC[case["prec"]])
        return s["y"]
    if op == "multi":
        m.matvec_multi(s["x"], s["y"], case["k"], PREC[case["prec"]])
        return s["y"]
    if op == "elasticity":
        m.matvec_elasticity(s["x"], s["y"])
        return s["y"]
    if op == "fem":
        m.rhs_quadrature(s["f"], s["b"])
        return {"load": s["b"], "error": m.l2_error(s["f"], s["u"])}
    if op == "transfer":
        t = s["transfers"][0]
        t.restrict(s["r"], s["c"], PREC[case["prec"]])
        t.prolong_add(s["e"], s["x"], s["y"], PREC[case["prec"]])
        return {"coarse": s["c"], "fine": s["y"]}
    if op == "vcycle":
        s["solver"].vcycle(s["b"], s["x"])
        return s["x"]
    if op == "solve":
        s["solver"].solve(s["b"], s["x"])
        return s["x"]
    s["solver"].solve_multi(s["b"], s["x"], case["k"])
    return s["x"]


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    damg = _hierarchy(case)
    info = [damg.info(l) for l in range(damg.nlevels)]
    op, F = case["op"], info[-1]
    size = 4 if case.get("prec") == "f32" else 8
    ncoef = {"helmholtz": 0, "kappa": 1, "kappa_mass": 2}[case.get("coef", "helmholtz")]
    mats = 1 if case.get("coef") == "kappa" else 2
    k = case.get("k", 1)

    def product(i, size, vectors, k=1):   # node list, type and level per element; coefficients; the vectors
        return (i.n_elem * (34 + ncoef * size) + vectors * i.n_node * size * k, 128.0 * mats * i.n_elem * k)

    def transfers(c, f, size, k=1):   # map of the fine nodes, coarse node lists, both vectors each way
        return 5 * f.n_node * 2 + 33 * c.n_elem + size * k * (3 * f.n_node + 2 * c.n_node), 32.0 * f.n_node * k

    def vcycle(size, k=1):
        b = fl = 0.0
        for l in range(1, len(info)):
            for pb, pf in [product(info[l], size, 4, k)] * 4 + [transfers(info[l - 1], info[l], size, k)]:
                b, fl = b + pb, fl + pf
        n0 = float(info[0].n_node)
        return b + n0 * n0 / 2 * size, fl + 2 * n0 * n0 * k

    if op in ("matvec", "multi"):
        b, fl = product(F, size, 2, k)
    elif op == "dirichlet":
        b, fl = product(F, size, 2)
        b += F.n_node
    elif op == "elasticity":
        b, fl = F.n_elem * 35 + F.n_node * 48, 2.0 * 576 * F.n_elem
    elif op == "fem":
        terms = {"cos": 3 * case["nfreq"], "gaussians": 8, "poly": 12}[case["fn"]]
        b = 2.0 * (F.n_elem * 50 + F.n_node * 8)
        fl = 2.0 * F.n_elem * 27 * (16 + terms)
    elif op == "transfer":
        b, fl = transfers(info[0], F, size)
    elif op == "vcycle":
        b, fl = vcycle(8)
    else:   # solves: about seven iterations, a product, a V-cycle and ten passes over the outer vectors each
        vb, vf = vcycle(4 if op == "solve_multi" else size, k)
        pb, pf = product(F, 8, 2, k)
        b, fl = 7 * (vb + pb + 10 * 8.0 * F.n_node * k), 7 * (vf + pf)
    return {"bytes": float(b), "flops": float(fl)}


# ---------------------------------------------------------------- the same in 64 bits, plain torch
# Vertex v of an element has bits (x, y, z).  In the frame of child 0 a hanging edge midpoint
# v = 1, 2, 4 is the mean of vertex 0 and the parent's vertex v, a hanging face centre
# v = 3, 5, 6 the mean of 0, the two edge vertices and v.
def _constraint():
    """P[mask][v][node]: value of vertex v from the values at the element's node list (child 0's frame)."""
    P = np.zeros((256, 8, 8))
    for mask in range(256):
        for v in range(8):
            nodes = [v]
            if mask >> v & 1 and 0 < v < 7:
                nodes = [0, v] if v in (1, 2, 4) else [0, v & -v, v & (v - 1), v]
            for q in nodes:
                P[mask, v, q] += 1.0 / len(nodes)
    return P


def _kron(ax):
    """K[i][j] = product over the axes of ax[axis][i's bit][j's bit]."""
    K = np.ones((8, 8))
    for i in range(8):
        for j in range(8):
            for a in range(3):
                K[i, j] *= ax[a][i >> a & 1][j >> a & 1]
    return K


_M1 = np.array([[2.0, 1.0], [1.0, 2.0]]) / 6.0
_K1 = np.array([[1.0, -1.0], [-1.0, 1.0]])
_C1 = np.array([[-0.5, -0.5], [0.5, 0.5]])   # integral of phi_i' phi_j


class _Level:
    """One mesh level on the GPU in 64 bits."""

    def __init__(self, damg, l, kappa=None, mass=None):
        L = damg.level(l)
        c = torch.as_tensor(L.child.astype(np.int64), device="cuda")
        H = torch.as_tensor(L.hnmask.astype(np.int64), device="cuda")
        nl = torch.as_tensor(L.nlist.astype(np.int64), device="cuda")
        v = torch.arange(8, device="cuda")
        self.perm = v[None, :] ^ c[:, None]                       # element vertex of child 0's vertex
        self.mask = (((H[:, None] >> self.perm) & 1) << v[None, :]).sum(1)
        self.nl = torch.gather(nl, 1, self.perm)                  # node list in child 0's frame
        self.nl_own, self.child = nl, c
        self.N, self.E = L.n_node, L.n_elem
        lev = torch.as_tensor(L.lev.astype(np.float64), device="cuda")
        self.h = 2.0 ** (1.0 - lev)
        self.anchor = torch.as_tensor(L.anchor.astype(np.float64), device="cuda") / 2.0 ** (L.max_depth - 1)
        self.P = torch.as_tensor(_constraint(), device="cuda")
        up = lambda a: torch.as_tensor(np.asarray(a, np.float64), device="cuda")
        self.kap = torch.ones_like(self.h) if kappa is None else up(kappa)
        self.mas = (torch.ones_like(self.h) if kappa is None else
                    torch.zeros_like(self.h) if mass is None else up(mass))
        lap = sum(_kron([_K1 if b == a else _M1 for b in range(3)]) for a in range(3))
        PT = self.P.transpose(1, 2).contiguous()
        self.L = PT @ up(lap) @ self.P
        self.M = PT @ up(_kron([_M1] * 3)) @ self.P

    def blocks(self):
        step = 1 << 18
        return [slice(i, min(i + step, self.E)) for i in range(0, self.E, step)]

    def matrix(self, sl):
        return ((self.kap * self.h)[sl, None, None] * self.L[self.mask[sl]] +
                (self.mas * self.h ** 3)[sl, None, None] * self.M[self.mask[sl]])

    def matvec(self, x):
        y = torch.zeros_like(x)
        for sl in self.blocks():
            nl = self.nl[sl]
            if x.dim() == 1:
                y.index_add_(0, nl.reshape(-1), (self.matrix(sl) * x[nl][:, None, :]).sum(2).reshape(-1))
                continue
            K = self.matrix(sl)
            for j0 in range(0, x.shape[1], 8):
                xe = x[:, j0:j0 + 8][nl]
                ye = sum(K[:, :, q, None] * xe[:, None, q, :] for q in range(8))
                y[:, j0:j0 + 8].index_add_(0, nl.reshape(-1), ye.reshape(-1, ye.shape[2]))
        return y

    def diagonal(self):
        d = torch.zeros(self.N, dtype=torch.float64, device="cuda")
        for sl in self.blocks():
            d.index_add_(0, self.nl[sl].reshape(-1), torch.diagonal(self.matrix(sl), dim1=1, dim2=2).reshape(-1))
        return d

    def dense(self):
        A = torch.zeros(self.N * self.N, dtype=torch.float64, device="cuda")
        for sl in self.blocks():
            nl = self.nl[sl]
            A.index_add_(0, (nl[:, :, None] * self.N + nl[:, None, :]).reshape(-1), self.matrix(sl).reshape(-1))
        return A.reshape(self.N, self.N)

    def elasticity(self, x, mu, lam):
        up = lambda a: torch.as_tensor(a, device="cuda")
        lap = sum(_kron([_K1 if b == a else _M1 for b in range(3)]) for a in range(3))
        K = {}
        for a in range(3):
            for b in range(3):   # integral of d_a phi_k d_b phi_j
                gd = _kron([_K1 if d == a == b else _C1 if d == a else _C1.T if d == b else _M1 for d in range(3)])
                K[a, b] = up((mu * lap if a == b else 0.0) + (mu + lam) * gd)
        y = torch.zeros_like(x)
        for sl in self.blocks():
            nl = self.nl[sl]
            P = self.P[self.mask[sl]]
            sign = 1.0 - 2.0 * ((self.child[sl, None] >> torch.arange(3, device="cuda")) & 1).double()
            xe = (P[:, :, :, None] * x[nl][:, None, :, :]).sum(2) * sign[:, None, :]   # mirrored to child 0
            z = torch.stack([sum((K[a, b][None] * xe[:, None, :, b]).sum(2) for b in range(3)) for a in range(3)], 2)
            ye = (P[:, :, :, None] * z[:, :, None, :]).sum(1) * (sign * self.h[sl, None])[:, None, :]
            y.index_add_(0, nl.reshape(-1), ye.reshape(-1, 3))
        return y

    def evaluate(self, case, X, Y, Z):
        if case["fn"] == "cos":
            k = torch.arange(1, case["nfreq"] + 1, device="cuda", dtype=torch.float64) * np.pi
            return ((1.0 + 3.0 * k * k) * torch.cos(k * X[..., None]) * torch.cos(k * Y[..., None]) *
                    torch.cos(k * Z[..., None])).sum(-1)
        if case["fn"] == "gaussians":
            r = torch.zeros_like(X)
            for mid, lo, hi, closed in ((0.1, 0.0, 0.2, False), (0.3, 0.2, 0.4, True), (0.6, 0.5, 0.7, True)):
                inside = torch.ones_like(X, dtype=torch.bool)
                for t in (X, Y, Z):
                    inside &= (t >= lo) & ((t <= hi) if closed else (t < hi))
                d2 = (X - mid) ** 2 + (Y - mid) ** 2 + (Z - mid) ** 2
                r += torch.where(inside, torch.exp(-d2 / 0.005), torch.zeros_like(r))
            return r
        c = _function(case).poly
        return (c[0] + c[1] * X + c[2] * Y + c[3] * Z + c[4] * X * Y + c[5] * Y * Z + c[6] * Z * X +
                c[7] * X * Y * Z)

    def load_and_error(self, case, u):
        g = np.sqrt(0.6)
        t = torch.tensor([0.0, g, -g], dtype=torch.float64, device="cuda")
        w = torch.tensor([8.0, 5.0, 5.0], dtype=torch.float64, device="cuda") / 9.0
        q = torch.cartesian_prod(t, t, t)
        wq = torch.cartesian_prod(w, w, w).prod(1)
        bits = (torch.arange(8, device="cuda")[:, None] >> torch.arange(3, device="cuda")) & 1
        phi = torch.where(bits[None] == 1, (1 + q[:, None, :]) / 2, (1 - q[:, None, :]) / 2).prod(2)   # [27][8]
        b = torch.zeros(self.N, dtype=torch.float64, device="cuda")
        err = 0.0
        inv = self.perm   # an involution: child 0's vertex of element vertex
        for sl in self.blocks():
            for s2 in [slice(i, min(i + (1 << 16), sl.stop)) for i in range(sl.start, sl.stop, 1 << 16)]:
                h, X = self.h[s2], self.anchor[s2, None, :] + self.h[s2, None, None] * (1 + q[None]) / 2
                f = self.evaluate(case, X[..., 0], X[..., 1], X[..., 2])
                P = self.P[self.mask[s2]]
                ph = phi[:, inv[s2]].permute(1, 0, 2)                       # shape functions in child 0's order
                ph = (ph[:, :, :, None] * P[:, None, :, :]).sum(2)          # [E][27][8], constrained
                fac = h ** 3 / 8.0
                nl = self.nl[s2]
                b.index_add_(0, nl.reshape(-1), (fac[:, None] * (f[:, :, None] * wq[None, :, None] * ph).sum(1)).reshape(-1))
                d = f - (ph * u[nl][:, None, :]).sum(2)
                err += float((fac * (wq * d * d).sum(1)).sum())
        return {"load": b, "error": float(np.sqrt(err))}


class _Transfer:
    """P and its transpose between two levels as (fine node, coarse node, weight) entries."""

    def __init__(self, damg, fine, coarse_level):
        C = coarse_level
        ce, pos = damg.transfer(fine)
        ce = torch.as_tensor(ce.astype(np.int64), device="cuda")
        pos = torch.as_tensor(pos.astype(np.int64), device="cuda")
        t = torch.stack([pos % 3, pos // 3 % 3, pos // 9], 1).double() / 2.0
        bits = (C.perm[ce][:, :, None] >> torch.arange(3, device="cuda")) & 1
        phi = torch.where(bits == 1, t[:, None, :], 1 - t[:, None, :]).prod(2)
        self.w = (phi[:, :, None] * C.P[C.mask[ce]]).sum(1)
        self.cn, self.Nc = C.nl[ce], C.N

    def up(self, c):
        if c.dim() == 1:
            return (self.w * c[self.cn]).sum(1)
        return sum(self.w[:, k, None] * c[self.cn[:, k]] for k in range(8))

    def down(self, f):
        c = torch.zeros((self.Nc,) + tuple(f.shape[1:]), dtype=torch.float64, device="cuda")
        for k in range(8):
            c.index_add_(0, self.cn[:, k], self.w[:, k] * f if f.dim() == 1 else self.w[:, k, None] * f)
        return c


class _Multigrid:
    def __init__(self, case, seed):
        damg = _hierarchy(case)
        coefs = _coefficients(case, damg, seed)
        self.lv = [_Level(damg, l, *coefs[l]) for l in range(damg.nlevels)]
        self.tr = [_Transfer(damg, l, self.lv[l - 1]) for l in range(1, damg.nlevels)]
        self.inv = [1.0 / L.diagonal() for L in self.lv]
        self.null = bool(_null_space(case))
        A = self.lv[0].dense()
        if self.null:
            A = A + A.trace() / (A.shape[0] ** 2)
        self.chol = torch.linalg.cholesky(A)

    def mean_free(self, v):
        return v - v.mean(0) if self.null else v

    def cycle(self, l, b):
        if l == 0:
            r = self.mean_free(b)
            return torch.cholesky_solve(r.reshape(r.shape[0], -1), self.chol).reshape(b.shape)
        L = self.lv[l]
        w = OMEGA * (self.inv[l] if b.dim() == 1 else self.inv[l][:, None])
        x = w * b
        x = x + w * (b - L.matvec(x))
        x = x + self.tr[l - 1].up(self.cycle(l - 1, self.tr[l - 1].down(b - L.matvec(x))))
        for _ in range(2):
            x = x + w * (b - L.matvec(x))
        return x

    def precondition(self, r):
        return self.mean_free(self.cycle(len(self.lv) - 1, r))

    def solve(self, b):
        """CG on every column to about 1e-13."""
        A = self.lv[-1].matvec
        r = self.mean_free(b.clone())
        x, z = torch.zeros_like(r), self.precondition(r)
        p, rz, b2 = z, (r * z).sum(0), (r * r).sum(0)
        for _ in range(60):
            w = A(p)
            a = rz / (p * w).sum(0)
            x, r = x + a * p, r - a * w
            if bool(((r * r).sum(0) <= 1e-26 * b2).all()):
                break
            z = self.precondition(r)
            rz, old = (r * z).sum(0), rz
            p = z + rz / old * p
        return self.mean_free(x)


def exact(case, seed):
    op = case["op"]
    if op in ("vcycle", "solve", "solve_multi"):
        mg = _Multigrid(case, seed)
        n = mg.lv[-1].N
        b = _uniform(seed, (n, case["k"]) if op == "solve_multi" else n, torch.float64)
        return mg.precondition(b) if op == "vcycle" else mg.solve(b)
    damg = _hierarchy(case)
    top = damg.nlevels - 1
    if op == "transfer":
        C, dt = _Level(damg, 0), DTYPE[case["prec"]]
        t, n = _Transfer(damg, 1, C), damg.info(1).n_node
        r, e, x = _uniform(seed, n, dt), _uniform(seed + 1, C.N, dt), _uniform(seed + 2, n, dt)
        return {"coarse": t.down(r.double()), "fine": x.double() + t.up(e.double())}
    F = _Level(damg, top, *_coefficients(case, damg, seed)[top])
    if op == "fem":
        return F.load_and_error(case, _uniform(seed, F.N, torch.float64))
    if op == "elasticity":
        return F.elasticity(_uniform(seed, (F.N, 3), torch.float64), 1.0, 1.5)
    if op == "multi":
        return F.matvec(_uniform(seed, (F.N, case["k"]), DTYPE[case["prec"]]).double())
    x = _uniform(seed, F.N, DTYPE[case["prec"]]).double()
    if op == "dirichlet":
        bdy = torch.as_tensor(damg.boundary(top), device="cuda") != 0
        return torch.where(bdy, x, F.matvec(torch.where(bdy, torch.zeros_like(x), x)))
    return F.matvec(x)
