"""The calls this framework is used for, at the sizes its users run them, as cases to time.

A case is a dict of plain values: `op`, what is called; `mesh` and its sizes, the block
table; `data`, the state on it; and the options of the call. `prepare` makes the plan and
the state on the GPU, `run` is one pass through the public entry points, `work` the bytes
and operations that pass cannot do without, `exact` what it returns in plain torch FP64.
"""
import functools
import itertools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dendro-gr_amd"))
import dgr  # noqa: E402
from dgr import workloads  # noqa: E402

DEV = "cuda"
PW = 3
SYM = [[0, 1, 2], [1, 3, 4], [2, 4, 5]]
PAIRS = [(0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2)]
BACKGROUND = [1.0, 1.0] + [0.0] * 10 + [1.0, 0.0, 0.0, 1.0, 0.0, 1.0] + [0.0] * 6
PUNCTURES = ((3.0, 0.0, 0.0), (-3.0, 0.0, 0.0))


# ------------------------------------------------------------------------------------------
# the cases

def listed():
    return [
        # one block through bssnrhs(), as a program that ports block by block calls it: the
        # smallest call, all launch and latency
        {"name": "rhs-block19-faces", "op": "rhs", "mesh": "ragged", "blocks": 1, "low": 19, "high": 19,
         "faces": 1.0, "data": "waves", "seed": 1},
        # one rank's share of a small run: blocks of odd and uneven sizes, some on the domain
        # boundary, with the curvature-adjusted dissipation
        {"name": "rhs-ragged-200", "op": "rhs", "mesh": "ragged", "blocks": 200, "low": 13, "high": 40,
         "faces": 0.3, "data": "waves", "seed": 2, "cako": True},
        # the other gauges of the reference's builds, all on, over an uneven octree
        {"name": "rhs-gauge-octree-2M", "op": "rhs", "mesh": "puncture", "scale": 0.03, "data": "punctures",
         "gauge": True},
        # a step of a 64-block grid with its outer boundary: what a test run or a strong-scaling
        # limit does, ten steps a call
        {"name": "rk4-small-64", "op": "rk4", "mesh": "refined", "base": 2, "top": 2, "data": "punctures",
         "refresh": "full", "nsteps": 10},
        # the uniform batch of the benchmark
        {"name": "rk4-uniform13-4096", "op": "rk4", "mesh": "uniform", "blocks": 4096, "data": "waves"},
        # the benchmark's uneven octree, 30.0 M points: the largest
        {"name": "rk4-octree-30M", "op": "rk4", "mesh": "puncture", "scale": 0.42, "data": "punctures"},
        # unigrid evolution: same-level neighbours refresh the padding at every stage
        {"name": "rk4-lattice13-4096", "op": "rk4", "mesh": "lattice", "nx": 16, "ny": 16, "nz": 16, "n": 13,
         "data": "waves", "refresh": "linked"},
        # production evolution: a 2:1 balanced octree with every padding refreshed across level jumps
        {"name": "rk4-refined-5M", "op": "rk4", "mesh": "refined", "base": 4, "top": 6, "data": "punctures",
         "refresh": "full"},
        # the same in mixed precision
        {"name": "rk4-refined-5M-mixed", "op": "rk4", "mesh": "refined", "base": 4, "top": 6, "data": "punctures",
         "refresh": "full", "precision": "mixed"},
        # the diagnostics written every few steps: all six constraints and the norm of the first
        {"name": "constraints-refined-5M", "op": "constraints", "mesh": "refined", "base": 4, "top": 6,
         "data": "punctures"},
        # unzip alone, before output or after a restart, on the deep octree (10.5 M points)
        {"name": "padding-refined-10M", "op": "padding", "mesh": "refined", "base": 4, "top": 9,
         "data": "punctures"},
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    op = rng.choice(["rhs", "rhs", "rk4", "rk4", "rk4", "constraints", "padding"])
    c = {"op": op}
    mesh = rng.choice({"rhs": ["ragged", "puncture", "uniform"], "constraints": ["ragged", "refined", "puncture"],
                       "rk4": ["puncture", "uniform", "lattice", "refined"], "padding": ["refined", "lattice"]}[op])
    c["mesh"] = mesh
    if mesh == "ragged":
        low = rng.randint(13, 30)
        c.update(blocks=spread(1, 800), low=low, high=low + rng.randint(0, 20), faces=rng.choice([0.0, 0.2, 1.0]),
                 seed=rng.randint(1, 999))
    elif mesh == "uniform":
        c.update(blocks=spread(16, 8000))
    elif mesh == "puncture":
        c.update(scale=round(math.exp(rng.uniform(math.log(0.002), math.log(0.25))), 4))
    elif mesh == "lattice":
        n, most = rng.choice([(13, 18), (19, 9), (25, 6)])
        c.update(n=n, nx=rng.randint(2, most), ny=rng.randint(2, most), nz=rng.randint(2, most))
    else:
        base = rng.randint(2, 4)
        c.update(base=base, top=base + rng.randint(0, 3))
    c["data"] = "punctures" if mesh in ("puncture", "refined") else "waves"
    if op == "rhs":
        c.update(cako=rng.random() < 0.3, gauge=rng.random() < 0.3)
    if op == "rk4":
        c["refresh"] = {"lattice": "linked", "refined": "full"}.get(mesh, "off")
        c["nsteps"] = rng.randint(1, 3)
        c["precision"] = rng.choice(["fp64"] * 5 + ["mixed"])
    return c


# ------------------------------------------------------------------------------------------
# what a program has in hand

@functools.lru_cache(maxsize=16)
def _table_of(key):
    c = dict(key)
    if c["mesh"] == "uniform":
        return workloads.uniform_13(c["blocks"])
    if c["mesh"] == "puncture":
        return workloads.puncture_octree(c["scale"])
    if c["mesh"] == "lattice":
        return workloads.lattice(shape=(c["nx"], c["ny"], c["nz"]), n=c["n"], h=0.05, origin=(-2.3, -1.9, -2.1),
                                 order="morton")
    if c["mesh"] == "refined":
        return workloads.refined_octree(c["base"], c["top"], 4.0)
    r = np.random.default_rng(c["seed"])  # ragged: sizes, spacings and boundary faces of a list of blocks
    t = np.zeros(c["blocks"], dtype=workloads.BLOCK_DTYPE)
    t["sz"] = r.integers(c["low"], c["high"], size=(len(t), 3), endpoint=True)
    n3 = np.prod(t["sz"].astype(np.uint64), axis=1)
    t["offset"] = np.concatenate([[0], np.cumsum(n3)[:-1]])
    on = r.random(len(t)) < c["faces"]
    t["bflag"] = np.where(on, 63 if len(t) == 1 else r.integers(1, 64, size=len(t)), 0)
    t["pmin"] = np.array([0.25, 0.05, -0.15]) + 4.0 * r.integers(0, 6, size=(len(t), 3))
    t["pmax"] = t["pmin"] + (t["sz"] - 1) * (0.1 / (1 + r.integers(0, 3, size=(len(t), 1))))
    return t


def _table(case):
    keys = ("mesh", "blocks", "scale", "nx", "ny", "nz", "n", "base", "top", "low", "high", "faces", "seed")
    return _table_of(tuple((k, case[k]) for k in keys if k in case))


def _groups(t, most=1 << 21):
    """Blocks of one size together, at most `most` padded points at a time: (block numbers, (nx, ny, nz))."""
    kinds, inverse = np.unique(t["sz"], axis=0, return_inverse=True)
    for k, sz in enumerate(kinds):
        every = np.nonzero(inverse.ravel() == k)[0]
        step = max(1, most // int(np.prod(sz.astype(np.int64))))
        for a in range(0, len(every), step):
            yield every[a:a + step], tuple(int(x) for x in sz)


def _columns(t, idx, sz):
    """Where the points of the blocks idx lie in a variable, [block, z, y, x]."""
    off = torch.from_numpy(t["offset"][idx].astype(np.int64)).to(DEV)
    n = sz[0] * sz[1] * sz[2]
    return (off[:, None] + torch.arange(n, device=DEV)).view(len(idx), sz[2], sz[1], sz[0])


def _geometry(t, idx, sz):
    """Spacings [3][block] and coordinates [3][block, z, y, x] (broadcast) of the blocks idx."""
    pmin = torch.from_numpy(t["pmin"][idx]).to(DEV)
    h = torch.from_numpy((t["pmax"][idx] - t["pmin"][idx]) / (t["sz"][idx] - 1.0)).to(DEV)
    x = []
    for a in range(3):
        line = pmin[:, a, None] + torch.arange(sz[a], device=DEV, dtype=torch.float64) * h[:, a, None]
        x.append(line.view([len(idx)] + [sz[a] if a == 2 - d else 1 for d in range(3)]))
    return [h[:, a].view(-1, 1, 1, 1) for a in range(3)], x


def _state(case, seed):
    """The state (24, points): smooth waves about flat space, or Brill-Lindquist punctures with noise."""
    t = _table(case)
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    u = torch.zeros((24, workloads.total_padded(t)), dtype=torch.float64, device=DEV)
    wave = torch.rand((24, 3, 5), generator=gen, dtype=torch.float64, device=DEV).cpu()
    for idx, sz in _groups(t):
        col = _columns(t, idx, sz).view(-1)
        _, x = _geometry(t, idx, sz)
        if case["data"] == "waves":
            for v in range(24):
                f = BACKGROUND[v]
                for a, k0, k1, k2, p in wave[v].tolist():
                    f = f + 1e-3 * (2 * a - 1) * torch.sin((1 + 3 * k0) * x[0] + (1 + 3 * k1) * x[1]
                                                           + (1 + 3 * k2) * x[2] + 6.28 * p)
                u[v, col] = f.reshape(-1)
            continue
        r = [torch.sqrt((x[0] - p[0]) ** 2 + (x[1] - p[1]) ** 2 + (x[2] - p[2]) ** 2) for p in PUNCTURES]
        psi = 1.0 + 0.25 / r[0] + 0.25 / r[1]
        u[0, col] = torch.clamp(psi ** -2, min=0.1).reshape(-1)
        u[1, col] = torch.clamp(psi ** -4, min=0.1).reshape(-1)
        u[12:18, col] = torch.tensor(BACKGROUND[12:18], dtype=torch.float64, device=DEV)[:, None]
        noise = torch.rand((24, len(col)), generator=gen, dtype=torch.float64, device=DEV)
        for v in list(range(2, 12)) + list(range(18, 24)):
            u[v, col] = 1e-6 * (2.0 * noise[v] - 1.0)
    return u


def _options(case):
    o = dict(ko_sigma=0.4)
    if case["mesh"] in ("uniform", "lattice", "ragged"):
        o.update(eta_central=2.0, eta_outer=2.0)
    if case.get("cako"):
        o.update(cako_enabled=1)
    if case.get("gauge"):
        # (the eta function is singular where chi passes through 1, as the waves do)
        o.update(eta_func=int(case["data"] == "punctures"), rochester=1, ssl=1, xi=(1.0, 1.0, 1.0))
    return o


T_RHS = 7.5  # the time the slow-start lapse reads


def _dt(t):
    return 0.25 * float(((t["pmax"] - t["pmin"]) / (t["sz"] - 1.0)).min())


def prepare(case, seed):
    t = _table(case)
    n = workloads.total_padded(t)
    s = {"op": case["op"], "plan": dgr.Plan(t, n), "u": _state(case, seed),
         "params": dgr.default_params(**_options(case))}
    if case["op"] == "rhs":
        s["out"] = torch.zeros_like(s["u"])
    elif case["op"] == "rk4":
        s["dt"], s["nsteps"] = _dt(t), case.get("nsteps", 1)
        s["plan"].set_precision(case.get("precision", "fp64"))
        s["plan"].set_halo_refresh({"off": 0, "linked": 1, "full": "full"}[case.get("refresh", "off")])
    elif case["op"] == "constraints":
        s["plan"].link_neighbors()
        s["out"] = torch.zeros((6, n), dtype=torch.float64, device=DEV)
    else:
        s["plan"].fill_sources()
    return s


def run(s):
    plan, u = s["plan"], s["u"]
    if s["op"] == "rhs":
        plan.rhs(s["out"], u, s["params"], t=T_RHS)
        return s["out"]
    if s["op"] == "rk4":
        plan.rk4_steps(u, s["dt"], s["params"], s["nsteps"])
        return u
    if s["op"] == "constraints":
        o = s["out"]
        plan.constraints(o[0], o[1:4], u, psi4=o[4:6])
        return o, plan.constraint_norm(o[0], r1=1.0, r2=1.0)
    plan.padding_fill(u)
    return u


def work(case):
    """Bytes: each padded state read once and each result written once; an RK4 stage also reads
    and writes the accumulator, reads the step's start and writes the next stage. Operations:
    6788 a point and right-hand side (first and second derivatives, dissipation, equations), 96 a
    stage update, about 2600 for the constraints (derivatives of 17 variables, no dissipation),
    2 x 7 a padding value."""
    t = _table(case)
    padded = float(np.prod(t["sz"].astype(np.float64), axis=1).sum())
    inner = float(np.prod(t["sz"].astype(np.float64) - 2 * PW, axis=1).sum())
    if case["op"] == "rhs":
        return {"bytes": 192 * padded + 192 * inner, "flops": 6788 * inner}
    if case["op"] == "rk4":
        stages = 4 * case.get("nsteps", 1)
        return {"bytes": stages * (192 * padded + 960 * inner), "flops": stages * 6884 * inner}
    if case["op"] == "constraints":
        return {"bytes": 192 * padded + (48 + 8) * inner, "flops": 2600 * inner}
    return {"bytes": 2 * 192 * (padded - inner), "flops": 14 * 24 * (padded - inner)}


# ------------------------------------------------------------------------------------------
# the same in plain torch, 64 bits

def _cut(f, a, lo, hi):
    """f from index lo to index hi along axis a (0 x, 1 y, 2 z)."""
    return f.narrow(3 - a, lo, hi - lo)


# rows of the one-sided closures at the three nodes next to a flagged low face: {offset: weight}
_D1_EDGE = [{0: -25, 1: 48, 2: -36, 3: 16, 4: -3}, {-1: -3, 0: -10, 1: 18, 2: -6, 3: 1}, {-2: 1, -1: -8, 1: 8, 2: -1}]
_D2_EDGE = [{0: 45, 1: -154, 2: 214, 3: -156, 4: 61, 5: -10}, {-1: 10, 0: -15, 1: -4, 2: 14, 3: -6, 4: 1},
            {-2: -1, -1: 16, 0: -30, 1: 16, 2: -1}]
_KO_EDGE = [({3: 1, 2: -3, 1: 3, 0: -1}, 59), ({3: 1, 2: -6, 1: 12, 0: -10, -1: 3}, 43),
            ({3: 1, 2: -6, 1: 15, 0: -19, -1: 12, -2: -3}, 49)]
_INNER = {"d1": ({-3: -1, -2: 9, -1: -45, 1: 45, 2: -9, 3: 1}, 60), "d2": ({-3: 2, -2: -27, -1: 270, 0: -490, 1: 270, 2: -27, 3: 2}, 180),
          "ko": ({-3: 1, -2: -6, -1: 15, 0: -20, 1: 15, 2: -6, 3: 1}, 64)}


def _stencil(f, a, h, lo, hi, kind):
    """d/da, d2/da2 or the dissipation along axis a; lo, hi: which blocks have that face flagged.
    The result has f's shape; its three outermost planes along a mean nothing."""
    n = f.shape[3 - a]
    scale = h * h if kind == "d2" else h
    w, den = _INNER[kind]
    out = torch.zeros_like(f)
    _cut(out, a, PW, n - PW).copy_(sum(c * _cut(f, a, PW + o, n - PW + o) for o, c in w.items()) / (den * scale))
    for side, on in ((1, lo), (-1, hi)):
        if not bool(on.any()):
            continue
        which = on.view(-1, 1, 1, 1)
        for r in range(3):
            at = PW + r if side > 0 else n - 1 - PW - r
            if kind == "ko":
                w, den = _KO_EDGE[r][0], 64.0 * _KO_EDGE[r][1] / 48.0
            else:
                w, den = (_D1_EDGE, _D2_EDGE)[kind == "d2"][r], 12.0
            sign = side if kind == "d1" else 1
            row = sum(sign * c * _cut(f, a, at + side * o, at + side * o + 1) for o, c in w.items()) / (den * scale)
            here = _cut(out, a, at, at + 1)
            here.copy_(torch.where(which, row, here))
    return out


class _Point:
    """Fields and derivatives at the interior points of a few blocks of one size."""

    def __init__(self, F, h, flags):
        self.F, self.h = F, h
        self.lo = [(flags >> (2 * a) & 1).bool() for a in range(3)]
        self.hi = [(flags >> (2 * a + 1) & 1).bool() for a in range(3)]
        self.first, self.second = {}, {}

    def inner(self, f):
        for a in range(3):
            f = _cut(f, a, PW, f.shape[3 - a] - PW)
        return f

    def f(self, v):
        return self.inner(self.F[v])

    def along(self, g, a, kind):
        return _stencil(g, a, self.h[a], self.lo[a], self.hi[a], kind)

    def d(self, a, v):
        if (v, a) not in self.first:
            self.first[v, a] = self.inner(self.along(self.F[v], a, "d1"))
        return self.first[v, a]

    def dd(self, a, b, v):
        a, b = min(a, b), max(a, b)
        if (v, a, b) not in self.second:
            g = self.along(self.F[v], a, "d2") if a == b else self.along(self.along(self.F[v], a, "d1"), b, "d1")
            self.second[v, a, b] = self.inner(g)
        return self.second[v, a, b]

    def ko(self, v):
        return sum(self.inner(self.along(self.F[v], a, "ko")) for a in range(3))


def _geometry_terms(p):
    """Inverse metric, Christoffel symbols and Ricci tensor of the conformal metric and of chi."""
    R3, R33 = range(3), list(itertools.product(range(3), repeat=2))
    g = [[p.f(12 + SYM[i][j]) for j in R3] for i in R3]
    co = [[g[(i + 1) % 3][(j + 1) % 3] * g[(i + 2) % 3][(j + 2) % 3] - g[(i + 1) % 3][(j + 2) % 3] * g[(i + 2) % 3][(j + 1) % 3]
           for j in R3] for i in R3]
    det = sum(g[0][j] * co[0][j] for j in R3)
    gu = [[co[j][i] / det for j in R3] for i in R3]
    dg = lambda k, i, j: p.d(k, 12 + SYM[i][j])  # noqa: E731
    first = [[[0.5 * (dg(j, k, i) + dg(i, k, j) - dg(k, i, j)) for j in R3] for i in R3] for k in R3]
    second = [[[sum(gu[k][m] * first[m][i][j] for m in R3) for j in R3] for i in R3] for k in R3]
    con = [sum(gu[i][j] * second[k][i][j] for i, j in R33) for k in R3]
    chi, dc = p.f(1), [p.d(a, 1) for a in R3]
    lap = sum(gu[k][m] * (p.dd(k, m, 1) - 1.5 * dc[k] * dc[m] / chi) for k, m in R33) - sum(con[m] * dc[m] for m in R3)
    ric = [[None] * 3 for _ in R3]
    for i, j in PAIRS:
        r = -0.5 * sum(gu[k][m] * p.dd(k, m, 12 + SYM[i][j]) for k, m in R33)
        r = r + 0.5 * sum(g[k][i] * p.d(j, 3 + k) + g[k][j] * p.d(i, 3 + k) for k in R3)
        r = r + 0.5 * sum(con[k] * (first[i][j][k] + first[j][i][k]) for k in R3)
        for m, n in R33:
            r = r + gu[m][n] * sum(second[k][m][i] * first[j][k][n] + second[k][m][j] * first[i][k][n]
                                   + second[k][i][n] * first[k][m][j] for k in R3)
        r = r + (p.dd(i, j, 1) - sum(second[k][i][j] * dc[k] for k in R3)) / (2 * chi) - dc[i] * dc[j] / (4 * chi * chi)
        ric[i][j] = ric[j][i] = r + g[i][j] * lap / (2 * chi)
    return g, gu, second, con, ric


def _equations(p, x, o, time):
    """The 24 right-hand sides at the interior points, without boundary values and dissipation."""
    R3, R33 = range(3), list(itertools.product(range(3), repeat=2))
    g, gu, ch, con, ric = _geometry_terms(p)
    al, chi, K = p.f(0), p.f(1), p.f(2)
    be, B = [p.f(6 + i) for i in R3], [p.f(9 + i) for i in R3]
    A = [[p.f(18 + SYM[i][j]) for j in R3] for i in R3]
    db = [[p.d(j, 6 + i) for j in R3] for i in R3]  # db[i][j] = d_j beta^i
    div = sum(db[i][i] for i in R3)
    da, dc, dK = ([p.d(a, v) for a in R3] for v in (0, 1, 2))
    adv = lambda v: sum(be[a] * p.d(a, v) for a in R3)  # noqa: E731
    out = [None] * 24
    up = [[sum(gu[i][k] * gu[j][m] * A[k][m] for k, m in R33) for j in R3] for i in R3]
    mixed = [[sum(gu[k][m] * A[m][j] for m in R3) for j in R3] for k in R3]
    dca = sum(gu[i][j] * dc[i] * da[j] for i, j in R33)
    hess = [[p.dd(i, j, 0) - sum(ch[k][i][j] * da[k] for k in R3) + (dc[i] * da[j] + dc[j] * da[i] - g[i][j] * dca) / (2 * chi)
             for j in R3] for i in R3]
    out[0] = adv(0) - 2 * al * K
    out[1] = adv(1) + (2.0 / 3.0) * chi * (al * K - div)
    out[2] = adv(2) - chi * sum(gu[i][j] * hess[i][j] for i, j in R33) + al * (K * K / 3 + sum(A[i][j] * up[i][j] for i, j in R33))
    X = [[al * ric[i][j] - hess[i][j] for j in R3] for i in R3]
    tr = sum(gu[i][j] * X[i][j] for i, j in R33)
    for i, j in PAIRS:
        lie = lambda M, v: (adv(v) + sum(M[i][k] * db[k][j] + M[k][j] * db[k][i] for k in R3)  # noqa: E731
                            - (2.0 / 3.0) * M[i][j] * div)
        out[12 + SYM[i][j]] = lie(g, 12 + SYM[i][j]) - 2 * al * A[i][j]
        out[18 + SYM[i][j]] = (lie(A, 18 + SYM[i][j]) + chi * (X[i][j] - g[i][j] * tr / 3)
                               + al * (K * A[i][j] - 2 * sum(A[i][k] * mixed[k][j] for k in R3)))
    if o.get("eta_func"):
        grad = sum(gu[i][j] * dc[i] * dc[j] for i, j in R33)
        eta = 1.31 * torch.sqrt(grad) * (1 - chi ** 2) ** -2
    else:
        r = torch.sqrt(x[0] ** 2 + x[1] ** 2 + x[2] ** 2)
        c, f = o.get("eta_central", 2.0), o.get("eta_outer", 0.25)
        eta = (c - f) * torch.exp(-(r / 40.0) ** 4) + f
    for i in R3:
        G = adv(3 + i) - sum(con[j] * db[i][j] for j in R3) + (2.0 / 3.0) * con[i] * div
        G = G + sum(gu[j][k] * p.dd(j, k, 6 + i) + gu[i][j] * p.dd(j, k, 6 + k) / 3 for j, k in R33)
        G = G - 2 * sum(up[i][j] * da[j] for j in R3) + 2 * al * sum(ch[i][j][k] * up[j][k] for j, k in R33)
        out[3 + i] = G - al * sum(3 * up[i][j] * dc[j] / chi + (4.0 / 3.0) * gu[i][j] * dK[j] for j in R3)
        if o.get("rochester"):
            out[6 + i] = o["xi"][1] * adv(6 + i) + 0.75 * o["xi"][2] * p.f(3 + i) - eta * be[i]
            out[9 + i] = torch.zeros_like(al)
        else:
            out[6 + i] = adv(6 + i) + 0.75 * B[i]
            out[9 + i] = out[3 + i] - eta * B[i] + adv(9 + i) - adv(3 + i)
    if o.get("ssl"):
        out[0] = out[0] - 0.6 * torch.sqrt(chi) * (al - torch.sqrt(chi)) * math.exp(-time * time / 800.0)
    return out


_FALLOFF = [1, 1, 1, 2, 2, 2] + [1] * 12 + [2] * 6


def _exact_rhs(t, u, o, time, out):
    """The right-hand sides of u's blocks into out's interior points."""
    for idx, sz in _groups(t, 1 << 20):
        col = _columns(t, idx, sz)
        h, x = _geometry(t, idx, sz)
        flags = torch.from_numpy(t["bflag"][idx].astype(np.int64)).to(DEV)
        p = _Point([u[v][col] for v in range(24)], h, flags)
        x = [_cut(x[a], a, PW, sz[a] - PW) for a in range(3)]
        k = _equations(p, x, o, time)
        face = torch.zeros_like(k[0], dtype=torch.bool)
        for a in range(3):
            for on, plane in ((p.lo[a], _cut(face, a, 0, 1)), (p.hi[a], _cut(face, a, face.shape[3 - a] - 1, face.shape[3 - a]))):
                plane |= on.view(-1, 1, 1, 1)
        r = torch.sqrt(x[0] ** 2 + x[1] ** 2 + x[2] ** 2)
        root = torch.sqrt(p.f(1)) if o.get("cako_enabled") else None
        to = p.inner(col)
        for v in range(24):
            if bool(face.any()):
                away = -(sum(x[a] * p.d(a, v) for a in range(3)) + _FALLOFF[v] * (p.f(v) - BACKGROUND[v])) / r
                k[v] = torch.where(face, away, k[v])
            sigma = o["ko_sigma"] if root is None else root * (0.99 if v == 0 or 6 <= v <= 11 else 0.3)
            out[v][to] = k[v] + sigma * p.ko(v)


def _enforced(S):
    """det(gt) = 1, tr(At) = 0, chi and alpha floored, on 24 values a point."""
    g, A = list(S[12:18]), list(S[18:24])
    det = lambda q: q[0] * (q[3] * q[5] - q[4] ** 2) - q[1] ** 2 * q[5] + 2 * q[1] * q[2] * q[4] - q[2] ** 2 * q[3]  # noqa: E731
    g = [q / det(g) ** (1.0 / 3.0) for q in g]
    d = det(g)
    gu = [g[3] * g[5] - g[4] ** 2, g[2] * g[4] - g[1] * g[5], g[1] * g[4] - g[2] * g[3], g[0] * g[5] - g[2] ** 2,
          g[1] * g[2] - g[0] * g[4], g[0] * g[3] - g[1] ** 2]
    tr = (A[0] * gu[0] + A[3] * gu[3] + A[5] * gu[5] + 2 * (A[1] * gu[1] + A[2] * gu[2] + A[4] * gu[4])) / (3 * d)
    A = [a - tr * q for a, q in zip(A, g)]
    return torch.stack([S[0].clamp(min=0.1), S[1].clamp(min=0.1), *S[2:12], *g, *A])


@functools.lru_cache(maxsize=2)
def _links_of(key):
    """For a lattice or an octree of equal blocks: level and cell of each block, a function that
    finds the block of a level and cell, and the 27 neighbours of each block's own level."""
    t = _table_of(key)
    m = int(t["sz"][0, 0]) - 2 * PW - 1
    h = (t["pmax"][:, 0] - t["pmin"][:, 0]) / (t["sz"][:, 0] - 1.0)
    corner = t["pmin"] + PW * h[:, None]
    level = np.rint(np.log2(h.max() / h)).astype(np.int64)
    cell = np.rint((corner - corner.min(axis=0)) / (m * h[:, None])).astype(np.int64)
    big = 1 << 14
    key_of = lambda L, c: ((L * big + c[..., 0]) * big + c[..., 1]) * big + c[..., 2]  # noqa: E731
    L, c = torch.from_numpy(level).to(DEV), torch.from_numpy(cell).to(DEV)
    keys, order = key_of(L, c).sort()

    def look(lev, at):
        k = key_of(lev, at)
        q = torch.searchsorted(keys, k).clamp(max=len(keys) - 1)
        return torch.where((keys[q] == k) & (at >= 0).all(-1) & (lev >= 0), order[q], -1)

    step = torch.tensor([[d % 3 - 1, d // 3 % 3 - 1, d // 9 - 1] for d in range(27)], device=DEV)
    nbr = look(L[:, None].expand(-1, 27), c[:, None] + step)
    nbr[:, 13] = -1
    return L, c, look, nbr


def _links(case):
    keys = ("mesh", "nx", "ny", "nz", "n", "base", "top")
    return _links_of(tuple((k, case[k]) for k in keys if k in case))


def _holder(look, L, at, m):
    """The lowest block of level L whose closed interior holds the node `at` (in that level's
    spacings): (block or -1, its cell)."""
    base = torch.div(at, m, rounding_mode="floor")
    best = torch.full(at.shape[:-1], 1 << 40, device=DEV)
    where = torch.zeros_like(base)
    for low in itertools.product((0, 1), repeat=3):
        off = torch.tensor(low, device=DEV)
        c = base - off
        b = look(L, c)
        good = (b >= 0) & ((off == 0) | (at == base * m)).all(-1) & (b < best)
        best = torch.where(good, b, best)
        where = torch.where(good[..., None], c, where)
    return torch.where(best < 1 << 40, best, -1), where


def _exact_fill(case, u, full):
    """Padding of u from the blocks that hold it: same level, then (full) finer nodes, then the
    order-6 interpolant of a coarser block's element."""
    t = _table(case)
    L, cell, look, nbr = _links(case)
    n = int(t["sz"][0, 0])
    m = n - 2 * PW - 1
    off = torch.from_numpy(t["offset"].astype(np.int64)).to(DEV)
    at = torch.tensor(list(itertools.product(range(n), repeat=3)), device=DEV).flip(1)  # x fastest
    way = (at >= n - PW).long() - (at < PW).long()
    pad = (way != 0).any(1)
    at, way = at[pad], way[pad]
    num = (way[:, 0] + 1) + 3 * (way[:, 1] + 1) + 9 * (way[:, 2] + 1)
    flat = lambda q: q[..., 0] + n * (q[..., 1] + n * q[..., 2])  # noqa: E731
    copies, inter = [], []
    for b0 in range(0, len(t), 1024):
        b = torch.arange(b0, min(b0 + 1024, len(t)), device=DEV)
        dst = off[b, None] + flat(at)
        src = nbr[b][:, num]
        here = src >= 0
        copies.append((dst[here], (off[src.clamp(min=0)] + flat(at - way * m))[here]))
        if not full:
            continue
        lev = L[b, None].expand(-1, len(at))
        node = cell[b, None] * m + at - PW
        left = ~here
        for rel in (0, 1, -1):  # same spacing, half, twice
            bl, lv, nd, ds = (q[left] for q in (b[:, None].expand(-1, len(at)), lev, node, dst))
            if rel < 0:  # an element holds the node at half steps
                hold, c = _holder(look, lv - 1, nd, 2 * m)
                got = hold >= 0
                inter.append((ds[got], hold[got], (nd - 2 * m * c)[got]))
            else:
                nd = nd * (1 + rel)
                hold, c = _holder(look, lv + rel, nd, m)
                hold = torch.where(hold == bl, -1, hold)
                got = hold >= 0
                copies.append((ds[got], (off[hold.clamp(min=0)] + flat(nd - c * m + PW))[got]))
            left[left.clone()] = ~got
    out = u.clone()
    for dst, src in copies:
        out[:, dst] = u[:, src]
    if inter and sum(len(q[0]) for q in inter):
        dst, hold, code = (torch.cat(q) for q in zip(*inter))
        el, which = torch.unique(hold, return_inverse=True)
        W = torch.tensor([[math.prod((0.5 * c - q) / (p - q) for q in range(7) if q != p) for p in range(7)] for c in range(13)],
                         dtype=torch.float64, device=DEV)
        inside = off[el, None] + flat(torch.tensor(list(itertools.product(range(PW, n - PW), repeat=3)), device=DEV).flip(1))
        for v in range(24):
            E = u[v][inside].view(-1, 7, 7, 7)
            for _ in range(3):  # the last axis each time, so that all three turn once
                E = (E @ W.T).permute(0, 3, 1, 2).contiguous()
            out[v, dst] = E[which, code[:, 2], code[:, 1], code[:, 0]]
    return out


def _exact_constraints(case, u):
    t = _table(case)
    out = torch.zeros((6, u.shape[1]), dtype=torch.float64, device=DEV)
    R3, R33 = range(3), list(itertools.product(range(3), repeat=2))
    linked = case["mesh"] in ("refined", "lattice")
    total, count = 0.0, 0
    for idx, sz in _groups(t, 1 << 20):
        col = _columns(t, idx, sz)
        h, x = _geometry(t, idx, sz)
        p = _Point([u[v][col] for v in range(24)], h, torch.from_numpy(t["bflag"][idx].astype(np.int64)).to(DEV))
        x = [_cut(x[a], a, PW, sz[a] - PW) for a in range(3)]
        g, gu, ch, con, ric = _geometry_terms(p)
        A = [[p.f(18 + SYM[i][j]) for j in R3] for i in R3]
        chi, K, dc = p.f(1), p.f(2), [p.d(a, 1) for a in R3]
        dA = lambda k, i, j: p.d(k, 18 + SYM[i][j])  # noqa: E731
        up = [[sum(gu[i][k] * gu[j][m] * A[k][m] for k, m in R33) for j in R3] for i in R3]
        to = p.inner(col)
        ham = chi * sum(gu[i][j] * ric[i][j] for i, j in R33) - sum(A[i][j] * up[i][j] for i, j in R33) + (2.0 / 3.0) * K * K
        out[0][to] = ham
        for i in R3:
            mom = sum(gu[j][k] * (dA(k, i, j) - sum(ch[m][k][i] * A[j][m] for m in R3) - 1.5 * A[k][i] * dc[j] / chi) for j, k in R33)
            out[1 + i][to] = mom - sum(p.f(3 + j) * A[i][j] for j in R3) - (2.0 / 3.0) * p.d(i, 2)
        # psi4 in the tetrad that Gram-Schmidt makes of r, theta and phi
        dot = lambda a, b: sum(g[i][j] * a[i] * b[j] for i, j in R33) / chi  # noqa: E731
        tetrad = []
        for e in ([x[0], x[1], x[2]], [x[0] * x[2], x[1] * x[2], -(x[0] ** 2 + x[1] ** 2)], [-x[1], x[0], 0 * x[2]]):
            along = [dot(q, e) for q in tetrad]
            e = [e[i] - sum(c * q[i] for c, q in zip(along, tetrad)) for i in R3]
            size = torch.sqrt(dot(e, e))
            tetrad.append([c / size for c in e])
        r, th, ph = tetrad
        Ar = [sum(A[i][j] * r[j] for j in R3) for i in R3]
        s = (sum(Ar[i] * r[i] for i in R3) + K * chi / 3 + 0.5 * sum(r[i] * dc[i] for i in R3)) / chi ** 2
        D = {(k, i, j): dA(j, k, i) + sum(ch[m][k][i] * A[m][j] for m in R3) for k in R3 for i, j in R33}
        re = im = 0.0
        for i, j in R33:
            mm, mn = th[i] * th[j] - ph[i] * ph[j], th[i] * ph[j] + th[j] * ph[i]
            rt, rp = th[i] * r[j] - th[j] * r[i], ph[i] * r[j] - ph[j] * r[i]
            U, V = (sum(e[k] * D[k, i, j] for k in R3) for e in (th, ph))
            re = re - 0.5 * (ric[i][j] + s * A[i][j]) * mm + 0.5 * (rt * U - rp * V) / chi
            im = im + 0.5 * (ric[i][j] + s * A[i][j]) * mn - 0.5 * (rp * U + rt * V) / chi
        tA, pA, tc, pc = (sum(e[i] * q[i] for i in R3) for q in (Ar, dc) for e in (th, ph))
        re = re + 0.5 * (tA * (tA + 0.5 * tc) - pA * (pA + 0.5 * pc)) / chi ** 2
        im = im - 0.5 * (tA * (pA + 0.5 * pc) + pA * (tA + 0.5 * tc)) / chi ** 2
        axis = ((x[0].abs() <= 1e-7) & (x[1].abs() <= 1e-7)).expand_as(re)
        out[4][to] = torch.where(axis, 0.0, re)
        out[5][to] = torch.where(axis, 0.0, im)
        # the norm: away from the punctures, each shared node at its lowest block
        keep = torch.ones_like(ham, dtype=torch.bool)
        for q in PUNCTURES:
            keep &= sum((x[a] - q[a]) ** 2 for a in range(3)).sqrt() >= 1.0
        if linked:
            nbr = _links(case)[3][torch.from_numpy(idx).to(DEV)]
            for d in range(27):
                lower = (nbr[:, d] >= 0) & (nbr[:, d] < torch.from_numpy(idx).to(DEV))
                part = keep
                for a, s_ in enumerate((d % 3 - 1, d // 3 % 3 - 1, d // 9 - 1)):
                    if s_:
                        part = _cut(part, a, *((0, 1) if s_ < 0 else (part.shape[3 - a] - 1, part.shape[3 - a])))
                part &= ~lower.view(-1, 1, 1, 1)
        total += float((ham[keep] ** 2).sum())
        count += int(keep.sum())
    return out, (math.sqrt(total / count) if count else -1.0)


def exact(case, seed):
    t = _table(case)
    padded = workloads.total_padded(t)
    if padded * (4 * case.get("nsteps", 1) if case["op"] == "rk4" else 1) > 140e6:
        return None  # minutes in plain torch
    u = _state(case, seed)
    o = _options(case)
    if case["op"] == "constraints":
        return _exact_constraints(case, u)
    if case["op"] == "padding":
        return _exact_fill(case, u, True)
    k = torch.zeros_like(u)
    if case["op"] == "rhs":
        _exact_rhs(t, u, o, T_RHS, k)
        return k
    refresh, dt = case.get("refresh", "off"), _dt(t)
    fill = (lambda s: s) if refresh == "off" else (lambda s: _exact_fill(case, s, refresh == "full"))
    inner = torch.zeros(padded, dtype=torch.bool, device=DEV)
    for idx, sz in _groups(t):
        inner[_Point([], None, torch.zeros(1, dtype=torch.int64)).inner(_columns(t, idx, sz)).reshape(-1)] = True
    inner = inner.nonzero().view(-1)
    for _ in range(case.get("nsteps", 1)):
        start = u[:, inner]
        s, total = u, start.clone()
        for weight, ahead in ((1 / 6, 0.5), (1 / 3, 0.5), (1 / 3, 1.0), (1 / 6, None)):
            s = fill(s)
            _exact_rhs(t, s, o, 0.0, k)
            total += weight * dt * k[:, inner]
            s = s.clone()
            s[:, inner] = _enforced(total if ahead is None else start + ahead * dt * k[:, inner])
        u = s
    return fill(u)
