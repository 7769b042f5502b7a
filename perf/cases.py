"""Timed cases of the CD3D / TCD3D path: what a program that calls parmoon_amd does.

A case is one call sequence of such a program, from a residual evaluation on
8^3 cells to the 2.1 million unknown solves of bench.py:

  defect     pmx_defect_noalloc on device vectors, r = b - A x and ||r||
  assemble   assembly of every level, then that residual with the new operator
  solve      assembly of every level, the preconditioned Krylov solve to an
             FP64 relative residual of 1e-12 and the download of the solution
  transient  initialisation and a few time steps with re-assembly, solution
  gradient   one training step of the smoother's network: loss and gradient

Sizes are those of bench.py, of the tests and of the shipped configurations;
meshes are powers of two by construction, the network's lattices are not.
``exact`` states the same results in FP64 with torch alone.
"""
import math

import numpy as np
import torch

import parmoon_amd as pa
from parmoon_amd import prm as P

TARGET = 1e-12  # relative FP64 residual of every solve
TAU = 1e-3      # step of the rotating transient (bench.py); the heat equation uses 0.1082532
_CTX = None


def _context():
    """One context (device and stream) for the program, as its systems share it."""
    global _CTX
    if _CTX is None:
        _CTX = pa.Context(0)
    return _CTX


def listed():
    return [
        # a residual evaluation on the smallest mesh of the tests: one call's latency
        dict(name="defect q1 8", kind="defect", order=1, nref=3, nref0=1, example="sine", eps=1e-3, linear=False),
        # the smoke check's problem: three small levels, everything launch-bound
        dict(name="solve q1 8 fp64", kind="solve", order=1, nref=3, nref0=1, example="sine", eps=1e-3, linear=False,
             precision=0, solver=16, smoother=3, omega=1.0, cycle=1),
        # the heat equation of the TCD3D program (amc.h): short steps on 16^3
        dict(name="heat q1 16 fp64", kind="transient", order=1, nref=4, nref0=1, example="heat", steps=6, linear=False,
             precision=0, omega=1.0),
        # the small SUPG configuration, 8^3..32^3 with the 8^3 level solved exactly
        dict(name="solve q1 32 fp64", kind="solve", order=1, nref=5, nref0=3, example="sine", eps=1e-3, linear=False,
             precision=0, solver=16, smoother=3, omega=1.0, cycle=1),
        # the default example (Laplace, Galerkin, 64-point rule) with another method: BiCGStab, W-cycles, SOR
        dict(name="solve q2 16 bicgstab", kind="solve", order=2, nref=4, nref0=1, example="laplace", eps=1.0,
             linear=False, precision=0, solver=13, smoother=2, omega=1.0, cycle=2),
        # a field of the log-normal set, FP32 inside FP64
        dict(name="solve q1 64 fp32", kind="solve", order=1, nref=6, nref0=2, example="lognormal", peclet=100.0,
             linear=False, precision=1, solver=16, smoother=3, omega=1.0, cycle=1),
        # a network training step on the 33^3 lattice of a level and on a ragged one
        dict(name="gradient 33", kind="gradient", M=33),
        # bench.py's operator: plain FP64, FP32 inside FP64, and with the learned smoother below the finest level
        dict(name="solve q2 64 fp64", kind="solve", order=2, nref=6, nref0=2, example="curl", eps=1e-4, linear=True,
             precision=0, solver=16, smoother=3, omega=1.0, cycle=1),
        dict(name="solve q2 64 fp32", kind="solve", order=2, nref=6, nref0=2, example="curl", eps=1e-4, linear=True,
             precision=1, solver=16, smoother=3, omega=1.0, cycle=1),
        dict(name="solve q2 64 learned", kind="solve", order=2, nref=6, nref0=2, example="curl", eps=1e-4, linear=True,
             precision=2, solver=16, smoother=3, omega=1.0, cycle=1, train=1200),
        # assembly with the reference's default rule (64 points) at full size
        dict(name="assemble q2 64", kind="assemble", order=2, nref=6, nref0=2, example="curl", eps=1e-4, linear=False),
        # bench.py --transient: 128^3 SUPG Crank-Nicolson, re-assembly in every step
        dict(name="rotating q1 128 fp32", kind="transient", order=1, nref=7, nref0=3, example="rotating", steps=3,
             linear=False, precision=1, omega=0.4),
    ]


def draw(rng):
    kind = rng.choice(["solve"] * 5 + ["transient", "transient", "assemble", "assemble", "defect", "gradient"])
    if kind == "gradient":
        return dict(kind=kind, M=int(round(math.exp(rng.uniform(math.log(9), math.log(65))))))
    order = rng.choice([1, 2])
    nref = rng.randint(3, 7) if order == 1 else rng.randint(2, 6)
    nref0 = min(nref - 1, rng.choice([1, 2, 3] if order == 1 else [1, 2]))
    c = dict(kind=kind, order=order, nref=nref, nref0=nref0, linear=rng.random() < 0.5)
    if kind == "transient":
        c["nref"] = nref = min(nref, 7 if order == 1 else 4)
        c.update(example=rng.choice(["rotating", "heat"]) if order == 1 else "heat", steps=rng.randint(1, 4),
                 precision=rng.choice([0, 1]))
        c["omega"] = 0.4 if c["example"] == "rotating" else 1.0
        c["nref0"] = min(nref - 1, nref0)
        return c
    c["example"] = rng.choice(["sine", "curl", "lognormal", "laplace"])
    if c["example"] == "lognormal":
        c["peclet"] = round(math.exp(rng.uniform(math.log(10), math.log(1000))), 3)
    else:
        c["eps"] = 1.0 if c["example"] == "laplace" else round(math.exp(rng.uniform(math.log(1e-4), math.log(1e-2))), 8)
        if c["example"] == "sine":
            c["eps"] = max(c["eps"], 1e-3)
    if kind == "solve":
        plain = c["example"] == "laplace"
        c.update(precision=rng.choice([0, 0, 1, 1, 3]), solver=rng.choice([16, 11, 13]) if plain else 16,
                 smoother=rng.choice([2, 3]) if plain else 3, omega=1.0, cycle=rng.choice([1, 1, 2]) if plain else 1)
    return c


# ---------------------------------------------------------------- inputs
def _block(case, seed):
    """The parameter block of a case: its example with the coefficients of the seed."""
    rng = np.random.default_rng(seed)
    ex = case["example"]
    if ex == "curl":
        p = P.config2(nref=3, seed=seed)
        p[P.EPS] = case["eps"]
    elif ex == "lognormal":
        p = P.lognormal(seed=seed, nref=case["nref"], peclet=case["peclet"])
    elif ex == "sine":
        p = P.config1b()
        p[P.EPS] = case["eps"]
        b = np.array([1.0, 2.0, 3.0]) + 0.3 * rng.standard_normal(3)
        p[P.B0:P.B2 + 1] = b / np.linalg.norm(b)
    elif ex == "laplace":
        p = P.base(P.EX_LAPLACE, eps=case["eps"] * rng.uniform(0.5, 2.0))
    elif ex == "heat":
        p = P.heat_amc(0.0)
    else:
        p = P.rotating(seed=seed, form=P.FORM_TCD_SUPG_AK)
    p[P.LINEAR] = 1.0 if case["linear"] else 0.0
    return p


def _step(case):
    """tau, theta1..theta4 of Crank-Nicolson."""
    return [TAU if case["example"] == "rotating" else 0.1082532, .5, .5, .5, .5]


def _initial(case, seed):
    """Initial values of the heat equation in the lattice's order: a few seeded modes."""
    rng = np.random.default_rng(seed)
    M = case["order"] * (1 << case["nref"]) + 1
    g = np.linspace(0.0, 1.0, M)
    u = np.zeros((M, M, M))
    for _ in range(6):
        k, a = rng.integers(1, 4, 3), rng.standard_normal()
        s = [np.sin(math.pi * kk * g) for kk in k]
        u += a * s[2][:, None, None] * s[1][None, :, None] * s[0][None, None, :]
    return u.reshape(-1)


def _vectors(case, seed, dev):
    """x and b of a residual evaluation (lattice order, FP64)."""
    M = case["order"] * (1 << case["nref"]) + 1
    g = torch.Generator(device="cpu").manual_seed(seed)
    return (torch.randn(M ** 3, dtype=torch.float64, generator=g).to(dev),
            torch.randn(M ** 3, dtype=torch.float64, generator=g).to(dev))


def _network(case, seed):
    """Weights (uniform, as an untrained network has them), input and target of a training step."""
    rng = np.random.default_rng(seed)
    M, w = case["M"], []
    for co, scale in ((16, 1.0), (16, 1.0), (16, 1.0), (1, 0.1)):
        a = math.sqrt(6.0 / (27 * 16)) * scale
        w += [rng.uniform(-a, a, co * 27 * 16), rng.uniform(-0.1, 0.1, co)]
    u = rng.standard_normal((M, M, M, 16), dtype=np.float32)
    u[..., 1:13] = 0.3 * u[..., 1:13] - 0.1  # couplings divided by the diagonal
    u[..., 13:] = 0.0
    return np.concatenate(w).astype(np.float32), u, rng.standard_normal((M, M, M), dtype=np.float32)


def _options(case):
    o = dict(restart=50 if case["kind"] == "transient" else 30 if case["order"] == 2 else 20, maxit=400,
             res_norm_min=0.0, red_factor=0.0, smoother=3, solver=16, cycle=1, rel_target=TARGET)
    o.update({k: case[k] for k in ("solver", "smoother", "omega", "cycle", "precision") if k in case})
    if case.get("train"):
        o.update(learned_levels=0, learned_skip=1, learned_steps=3, learned_pre=1)
    return P.solver_opt(**o)


def prepare(case, seed):
    ctx = _context()
    kind = case["kind"]
    if kind == "gradient":
        S = pa.System(ctx, 1, 2, 1)  # the networks belong to a system; the lattice is the caller's
        w, u, t = _network(case, seed)
        S.learned_params(w)
        return dict(case=case, S=S, u=u, t=t)
    S = pa.System(ctx, case["nref0"], case["nref"] - case["nref0"] + 1, case["order"])
    st = dict(case=case, S=S, prm=_block(case, seed))
    if kind in ("defect", "assemble"):
        st["x"], st["b"] = _vectors(case, seed, "cuda")
        st["r"], st["res"] = torch.empty_like(st["b"]), torch.empty(1, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        if kind == "defect":
            S.assemble(st["prm"])
        return st
    st["opt"] = _options(case)
    if kind == "transient":
        st["td"] = _step(case)
        st["sol0"] = None
        if case["example"] == "heat":
            bi, gn = S.numbering()
            lat = _cells_lattice(case["nref"], case["order"]).reshape(-1)
            st["sol0"] = np.empty(int(S.dims()[0]))
            st["sol0"][gn] = _initial(case, seed)[lat]
    if case.get("train"):
        S.assemble(st["prm"])
        S.learned_train(P.solver_opt(**dict(solver=16, restart=30, maxit=400, res_norm_min=0.0, smoother=3, omega=1.0,
                                            precision=1)),
                        samples=32, steps=case["train"], lr=2e-3, seed=1, levels=0, data=1, skip=1)
    return st


def run(state):
    case, S = state["case"], state["S"]
    kind = case["kind"]
    if kind == "gradient":
        g, loss = S.learned_gradient(state["u"], state["t"])
        return dict(grads=g, loss=loss)
    if kind in ("defect", "assemble"):
        if kind == "assemble":
            S.assemble(state["prm"])
        S.defect_noalloc(state["x"].data_ptr(), state["b"].data_ptr(), state["r"].data_ptr(), state["res"].data_ptr())
        return dict(r=state["r"], res=state["res"])
    if kind == "solve":
        S.assemble(state["prm"])
        S.solve_resident(state["opt"])
        return S.solution()
    S.tcd_init(state["prm"], state["sol0"])
    p = state["prm"].copy()
    for m in range(case["steps"]):
        p[P.TIME] = (m + 1) * state["td"][0]
        S.tcd_step(p, state["td"], state["opt"])
    return S.solution()


# ---------------------------------------------------------------- what a pass cannot do without
def _sizes(case):
    n, o = 1 << case["nref"], case["order"]
    M = o * n + 1
    row = sum((5 if x % 2 == 0 else 3) if o == 2 else 3 for x in range(1, M - 1))
    nnz = row ** 3 + M ** 3 - (M - 2) ** 3
    deg = (2 if case["linear"] else 3) * o
    nq = (2 if deg <= 2 else 3 if deg <= 5 else 4) ** 3
    return n ** 3, M ** 3, nnz, nq, (o + 1) ** 3


def work(case):
    """Each operator entry written once by an assembly and read once by a product, each vector once."""
    if case["kind"] == "gradient":
        N = case["M"] ** 3
        return {"bytes": 4.0 * (17 * N + 2 * 21217), "flops": 3 * 2.0 * 27 * N * (3 * 256 + 16)}
    cells, N, nnz, nq, nb = _sizes(case)
    asm = cells * nq * (8.0 * nb * nb + 32 * nb)
    product = dict(bytes=8.0 * (nnz + 3 * N), flops=2.0 * nnz)
    if case["kind"] == "defect":
        return product
    if case["kind"] in ("assemble", "solve"):
        return {"bytes": product["bytes"] + 8.0 * (nnz + N), "flops": product["flops"] + asm}
    steps = case["steps"]
    return {"bytes": steps * (product["bytes"] + 16.0 * nnz) + 8.0 * nnz, "flops": steps * (product["flops"] + asm)}


# ---------------------------------------------------------------- the same in FP64, with torch alone
def _cells_lattice(nref, order):
    """Lattice index of the local nodes of every cell, in the order of the reference's cells and
    local nodes (depth first through the regular refinement, each child with its own axes)."""
    axes = [(1, 2, 3), (2, -1, 3), (-1, -2, 3), (-2, 1, 3), (2, 1, -3), (-1, 2, -3), (-2, -1, -3), (1, -2, -3)]
    corner = [(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1)]
    o, e = np.zeros((1, 3), np.int64), np.eye(3, dtype=np.int64)[None]
    size = 1 << nref
    while size > 1:
        os, es = [], []
        for j in range(8):
            os.append(o + size * np.einsum("a,cad->cd", np.array(corner[j]), e))
            es.append(np.stack([np.sign(c) * e[:, abs(c) - 1] for c in axes[j]], 1))
        o, e = np.stack(os, 1).reshape(-1, 3), np.stack(es, 1).reshape(-1, 3, 3)
        size //= 2
    k = order + 1
    loc = np.array([(a, b, c) for c in range(k) for b in range(k) for a in range(k)])
    X = order * o[:, None, :] + np.einsum("ja,cad->cjd", loc, e)
    M = order * (1 << nref) + 1
    return X[..., 0] + M * (X[..., 1] + M * X[..., 2])


def _dof_lattice(nref, order):
    """Lattice index of every degree of freedom: first encounter, interior nodes before Dirichlet nodes."""
    lat = _cells_lattice(nref, order).reshape(-1)
    M = order * (1 << nref) + 1
    nodes, first = np.unique(lat, return_index=True)
    nodes = nodes[np.argsort(first)]
    x, y, z = nodes % M, nodes // M % M, nodes // (M * M)
    bd = (x == 0) | (y == 0) | (z == 0) | (x == M - 1) | (y == M - 1) | (z == M - 1)
    return np.concatenate([nodes[~bd], nodes[bd]])


class _Space:
    """Cells, rule and basis tables of the unit cube refined nref times, on torch."""

    def __init__(self, case, dev):
        self.n, self.o, self.dev = 1 << case["nref"], case["order"], dev
        n, o = self.n, self.o
        self.M = o * n + 1
        self.h = 1.0 / n
        deg = (2 if case["linear"] else 3) * o
        x1, w1 = np.polynomial.legendre.leggauss(2 if deg <= 2 else 3 if deg <= 5 else 4)
        if o == 1:
            v, d = np.stack([(1 - x1) / 2, (1 + x1) / 2], 1), np.stack([-0.5 + 0 * x1, 0.5 + 0 * x1], 1)
        else:
            v = np.stack([x1 * (x1 - 1) / 2, 1 - x1 * x1, x1 * (x1 + 1) / 2], 1)
            d = np.stack([x1 - 0.5, -2 * x1, x1 + 0.5], 1)
        kron = lambda z, y, x: np.kron(np.kron(z, y), x)  # noqa: E731  (x fastest, points and nodes)
        T = lambda a: torch.tensor(a, dtype=torch.float64, device=dev)  # noqa: E731
        g = 2.0 * n
        self.phi = [T(kron(v, v, v)), T(g * kron(v, v, d)), T(g * kron(v, d, v)), T(g * kron(d, v, v))]  # [q, node]
        self.w = T(kron(w1[:, None], w1[:, None], w1[:, None])[:, 0]) * (self.h ** 3 / 8)
        c = torch.arange(n ** 3, device=dev)
        cz, cy, cx = c // (n * n), c // n % n, c % n
        q = np.array([(a, b, e) for e in x1 for b in x1 for a in x1])
        at = lambda i, k: (i.double()[:, None] + 0.5 * (1 + T(q[:, k]))[None]) * self.h  # noqa: E731
        self.X, self.Y, self.Z = at(cx, 0), at(cy, 1), at(cz, 2)
        loc = torch.tensor([a + self.M * (b + self.M * e) for e in range(o + 1) for b in range(o + 1)
                            for a in range(o + 1)], device=dev)
        self.idx = (o * cx + self.M * (o * cy + self.M * (o * cz)))[:, None] + loc[None]
        p = torch.arange(self.M ** 3, device=dev)
        pz, py, px = p // (self.M ** 2), p // self.M % self.M, p % self.M
        e = self.M - 1
        self.bd = (px == 0) | (py == 0) | (pz == 0) | (px == e) | (py == e) | (pz == e)
        self.nodes = px.double() / e, py.double() / e, pz.double() / e

    def rows(self, q):
        """sum over cells of local vectors [cell, node]."""
        y = torch.zeros(self.M ** 3, dtype=torch.float64, device=self.dev)
        return y.index_add_(0, self.idx.reshape(-1), q.reshape(-1))

    def matrix(self, D):
        """Local matrices of sum_q sum_(e,d) D[e, d](cell, q) phi_e,a phi_d,b."""
        nb = self.idx.shape[1]
        K = torch.zeros(self.n ** 3, nb * nb, dtype=torch.float64, device=self.dev)
        for (e, d), c in D.items():
            K += c @ (self.phi[e][:, :, None] * self.phi[d][:, None, :]).reshape(-1, nb * nb)
        return K.reshape(-1, nb, nb)

    def load(self, r):
        return self.rows(sum(c @ self.phi[e] for e, c in r.items()))

    def times(self, K, x):
        """A x of the interior rows."""
        y = self.rows(torch.bmm(K, x[self.idx].unsqueeze(2)).squeeze(2))
        return torch.where(self.bd, torch.zeros_like(y), y)


def _coefficients(prm, s, t):
    """eps, b, c, f at the points of every cell."""
    ex, X, Y, Z, pi = int(prm[P.EXAMPLE]), s.X, s.Y, s.Z, math.pi
    zero = torch.zeros_like(X)
    eps = zero + float(prm[P.EPS])
    b = [zero + float(v) for v in prm[P.B0:P.B2 + 1]]
    if ex == P.EX_LAPLACE:
        return eps, [zero] * 3, 3 * pi * pi * eps * torch.sin(pi * X) * torch.sin(pi * Y) * torch.sin(pi * Z)
    if ex == P.EX_SINE_CD:
        sx, sy, sz = (torch.sin(pi * v) for v in (X, Y, Z))
        cx, cy, cz = (torch.cos(pi * v) for v in (X, Y, Z))
        return eps, b, 3 * pi * pi * eps * sx * sy * sz + pi * (b[0] * cx * sy * sz + b[1] * sx * cy * sz
                                                               + b[2] * sx * sy * cz)
    if ex == P.EX_HEAT_AMC:
        return zero + 1.0, [zero] * 3, ((3 * pi * pi - 0.1) * math.exp(-0.1 * t) * torch.sin(pi * X)
                                        * torch.cos(pi * Y) * torch.cos(pi * Z))
    if ex == P.EX_ROTATING:
        return eps, [-(Y - 0.5), X - 0.5, zero + 0.2], zero
    if ex == P.EX_LOGNORMAL:
        G = sum(torch.cos(float(g[0]) * X + float(g[1]) * Y + float(g[2]) * Z + float(g[3]))
                for g in prm[P.GRF:P.GRF + 256].reshape(64, 4))
        return eps * torch.exp(float(prm[P.GRF_SIGMA]) * math.sqrt(2.0 / 64) * G), b, zero + 1.0
    dA = [[zero.clone() for _ in range(3)] for _ in range(3)]
    for c, modes in enumerate(prm[P.FOURIER:P.FOURIER + 120].reshape(3, 8, 5)):
        for a, kx, ky, kz, ph in modes.tolist():
            cs = 2 * pi * a * torch.cos(2 * pi * (kx * X + ky * Y + kz * Z) + ph)
            for d, k in enumerate((kx, ky, kz)):
                dA[c][d] += k * cs
    sc = float(prm[P.BSCALE])
    return eps, [sc * (dA[2][1] - dA[1][2]), sc * (dA[0][2] - dA[2][0]), sc * (dA[1][0] - dA[0][1])], zero + 1.0


def _delta(prm, s, eps, b, v=1.0):
    """The streamline parameter (SDFEM_TYPE 2) of the coefficients times v, times v."""
    hK = math.sqrt(3.0) * s.h
    nb = v * torch.sqrt(b[0] ** 2 + b[1] ** 2 + b[2] ** 2)
    al = nb * hK / (2 * v * eps)
    dl = hK * (1 / torch.tanh(al) - 1 / al) / (2 * nb)
    return float(prm[P.DELTA0]) * v * torch.where(nb > 0, dl, torch.zeros_like(dl))


def _convection_diffusion(s, eps, b, f, dl):
    """Local matrices and load of (eps grad u, grad v) + (b.grad u, v + delta b.grad v) = (f, v + delta b.grad v)."""
    D = {(0, d + 1): s.w * b[d] for d in range(3)}
    for e in range(3):
        for d in range(3):
            D[e + 1, d + 1] = s.w * ((eps if e == d else 0.0) + dl * b[e] * b[d])
    r = {0: s.w * f}
    r.update({e + 1: s.w * f * dl * b[e] for e in range(3)})
    return s.matrix(D), s.load(r)


def _boundary(prm, s, t):
    x, y, z = s.nodes
    pi = math.pi
    ex = int(prm[P.EXAMPLE])
    if ex in (P.EX_LAPLACE, P.EX_SINE_CD):
        return torch.sin(pi * x) * torch.sin(pi * y) * torch.sin(pi * z)
    if ex == P.EX_HEAT_AMC:
        return math.exp(-0.1 * t) * torch.sin(pi * x) * torch.cos(pi * y) * torch.cos(pi * z)
    return torch.zeros_like(x)


def _steady(prm, s):
    eps, b, f = _coefficients(prm, s, 0.0)
    supg = int(prm[P.FORM]) == P.FORM_SDFEM
    K, F = _convection_diffusion(s, eps, b, f, _delta(prm, s, eps, b) if supg else torch.zeros_like(f))
    return K, torch.where(s.bd, _boundary(prm, s, 0.0), F)


def _gmres(A, b, most):
    """A x = b by full GMRES, twice (the second on the residual of the first); None if it takes over `most` steps."""
    x = torch.zeros_like(b)
    bn = float(b.norm())
    if bn == 0.0:
        return x
    for _ in range(3):
        r = b - A(x)
        beta = float(r.norm())
        if beta <= 2e-15 * bn:
            break
        V = torch.empty(min(most, 64) + 1, b.numel(), dtype=b.dtype, device=b.device)
        V[0] = r / beta
        H, rot, g = [], [], [beta]
        while True:
            k = len(H)
            if k >= most:
                return None
            if k + 2 > V.shape[0]:
                V = torch.cat([V, torch.empty_like(V)])
            w = A(V[k])
            h = V[:k + 1] @ w
            w -= h @ V[:k + 1]
            h2 = V[:k + 1] @ w
            w -= h2 @ V[:k + 1]
            nw = float(w.norm())
            V[k + 1] = w / nw
            c = (h + h2).tolist() + [nw]
            for i, (cs, sn) in enumerate(rot):
                c[i], c[i + 1] = cs * c[i] + sn * c[i + 1], -sn * c[i] + cs * c[i + 1]
            d = math.hypot(c[k], c[k + 1])
            rot.append((c[k] / d, c[k + 1] / d))
            g.append(-rot[k][1] * g[k])
            g[k] *= rot[k][0]
            H.append(c[:k] + [d])
            if abs(g[-1]) <= 1e-9 * beta or abs(g[-1]) <= 1e-15 * bn:
                break
        k = len(H)
        y = np.zeros(k)
        for i in range(k - 1, -1, -1):
            y[i] = (g[i] - sum(H[j][i] * y[j] for j in range(i + 1, k))) / H[i][i]
        x = x + torch.tensor(y, dtype=b.dtype, device=b.device) @ V[:k]
        del V
    return x


def _solve(s, K, rhs, most):
    """The interior rows of K with the Dirichlet values of rhs, scaled by the diagonal."""
    diag = s.rows(torch.diagonal(K, dim1=1, dim2=2))
    g = torch.where(s.bd, rhs, torch.zeros_like(rhs))
    inner = ~s.bd
    at = torch.nonzero(inner).squeeze(1)
    dg = diag[at]

    def A(v):
        x = torch.zeros_like(rhs)
        x[at] = v / dg
        return s.times(K, x)[at]

    v = _gmres(A, (rhs - s.times(K, g))[at], most)
    if v is None:
        return None
    g[at] = v / dg
    return g


def _transient(case, prm, s, seed):
    td = _step(case)
    tau, th1, th2, th3, th4 = td
    zero = torch.zeros_like(s.X)
    Mm = s.matrix({(0, 0): s.w + zero})
    eps, b, f = _coefficients(prm, s, 0.0)
    old = s.load({0: s.w * f})
    if case["example"] == "heat":
        u = torch.tensor(_initial(case, seed), device=s.dev)
    else:
        B = prm[P.BLOB:P.BLOB + 4].tolist()
        u = torch.exp(-sum((x - c) ** 2 for x, c in zip(s.nodes, B)) / (2 * B[3] ** 2))
    u = torch.where(s.bd, _boundary(prm, s, 0.0), u)
    for m in range(case["steps"]):
        t = (m + 1) * tau
        eps, b, f = _coefficients(prm, s, t)
        if case["example"] == "heat":
            A, F = _convection_diffusion(s, eps, b, f, zero)
            MK = Mm
        else:
            dl = _delta(prm, s, eps, b, th1 * tau)
            A, F = _convection_diffusion(s, eps, b, f, dl)
            MK = Mm + s.matrix({(e + 1, 0): s.w * dl * b[e] for e in range(3)})
        g = _boundary(prm, s, t)
        rhs = tau * th3 * old + tau * th4 * F + s.times(MK, u) - tau * th2 * s.times(A, u)
        u = _solve(s, MK + tau * th1 * A, torch.where(s.bd, g, rhs), 600)
        if u is None:
            return None
        old = F
    return u


def _network_exact(case, seed, dev):
    w, u, t = _network(case, seed)
    M = case["M"]
    p = torch.tensor(w.astype(np.float64), device=dev, requires_grad=True)
    a = torch.tensor(u.astype(np.float64), device=dev)
    k = 0
    for layer, co in enumerate((16, 16, 16, 1)):
        W = p[k:k + co * 432].reshape(co, 27, 16)
        bias = p[k + co * 432:k + co * 433]
        k += co * 433
        pad = torch.nn.functional.pad(a, (0, 0, 1, 1, 1, 1, 1, 1))
        a = bias + sum(pad[q // 9:q // 9 + M, q // 3 % 3:q // 3 % 3 + M, q % 3:q % 3 + M] @ W[:, q].t()
                       for q in range(27))
        if layer < 3:
            a = 0.5 * a * (1 + torch.erf(a / math.sqrt(2.0)))
    d = (a[..., 0] - torch.tensor(t.astype(np.float64), device=dev))[1:-1, 1:-1, 1:-1]
    loss = (d * d).sum() / (M - 2) ** 3
    loss.backward()
    return dict(grads=p.grad.cpu().numpy(), loss=float(loss.detach()))


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if case["kind"] == "gradient":
        return _network_exact(case, seed, dev)
    prm = _block(case, seed)
    s = _Space(case, dev)
    if case["kind"] == "transient":
        u = _transient(case, prm, s, seed)
    else:
        K, rhs = _steady(prm, s)
        if case["kind"] in ("defect", "assemble"):
            x, b = _vectors(case, seed, dev)
            r = b - torch.where(s.bd, x, s.times(K, x))
            return dict(r=r, res=r.norm().reshape(1))
        # (the unrestarted vectors of the 2.1 million unknown solves take too long)
        u = _solve(s, K, rhs, 900) if s.M ** 3 < 10 ** 6 else None
    return None if u is None else u[torch.from_numpy(_dof_lattice(case["nref"], case["order"])).to(dev)].cpu().numpy()
