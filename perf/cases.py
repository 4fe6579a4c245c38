"""The workloads by which the speed of this framework is judged, through its public entry points.

A case is one call (or one short sequence of calls) that a DQMC program makes again and again:
sweeps of one chain from the smallest lattice to the largest, many chains together, the request
loop, the stack build, replaying recorded configurations, global updates and the two kinds of
measurement.  Lattices, couplings and chain counts are those of the benchmark and the tests:
the 4x4 chain of the fixtures, the 16x16 headline chain, the 24x24 attractive chain, the
64-chain batch and the request mix, and odd sizes between them.

Everything runs in FP64.  The mixed-precision form is left out: at these couplings it exceeds
its own bound and its calls raise.  Couplings stay at |U| <= 4, where the Green's function
propagated between two stabilisations keeps about nine digits, so that the accepted flips do
not hang on the rounding of one implementation.
"""
import importlib.util
import math
import os
import random
import sys

import numpy as np

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DTAU = 0.1


def _pkg():
    """The package (its folder's name is not a Python identifier)."""
    name = "montecarlo_jl_amd"
    if name not in sys.modules:
        d = os.path.join(_ROOT, "montecarlo.jl_amd")
        spec = importlib.util.spec_from_file_location(name, os.path.join(d, "__init__.py"),
                                                      submodule_search_locations=[d])
        sys.modules[name] = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(sys.modules[name])
    return sys.modules[name]


# ---- the cases -----------------------------------------------------------------------------
def _case(name, kind, lattice="square", L=4, U=4.0, mu=0.0, slices=40, safe_mult=10, **more):
    """U in the reference's convention: negative is repulsive (magnetic field, two flavours)."""
    return dict(name=name, kind=kind, lattice=lattice, L=L, U=U, mu=mu, slices=slices,
                safe_mult=safe_mult, **more)


def listed():
    return [
        # equal-time observables of the headline chain, once per measured sweep: the smallest
        # call a run makes, all latency
        _case("equal_time_16x16", "equal_time", L=16, U=-4.0, slices=20),
        # one sweep and its Green's function: the fixture chain, where launches count most
        _case("sweep_4x4", "sweep", L=4, U=4.0, slices=40),
        # an odd ragged one: 98 sites, 55 slices in chunks of 9 and 10, two flavours
        _case("sweep_honeycomb_7", "sweep", "honeycomb", 7, U=-3.0, slices=55),
        # the headline chain: 16x16, beta = 10, two flavours
        _case("sweep_16x16", "sweep", L=16, U=-4.0, slices=100),
        # the 24x24 attractive chain, beta = 12, away from half filling
        _case("sweep_24x24", "sweep", L=24, U=4.0, mu=-0.5, slices=120),
        # the largest square lattice of the request mix, two flavours, at a high temperature
        _case("sweep_32x32", "sweep", L=32, U=-4.0, slices=40),
        # 64 independent small chains swept together: a parameter scan on one GPU
        _case("batch_64", "batch", L=16, U=-4.0, slices=100, chains=64, mix=2024),
        # eight requests through the serving loop: admission, stack build, one sweep, result
        _case("serve_8", "serve", L=12, U=-4.0, slices=80, chains=8, mix=7),
        # a new configuration's stack and Green's function (admission, restart): 225 sites, long
        _case("build_15x15", "build", L=15, U=-4.0, slices=200),
        # one recorded configuration replayed: field in, Green's function from scratch out
        _case("replay_12x12", "replay", L=12, U=-2.0, slices=80, at=0),
        # a measuring sweep with the charge susceptibility (the imaginary-time integral)
        _case("susceptibility_8x8", "susceptibility", L=8, U=-4.0, slices=50, observable="charge"),
        # a global update: a proposal's weight from scratch, its stack if it is accepted
        _case("global_10x10", "global", L=10, U=4.0, slices=60, flips=3),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _lattice(rng, lo, hi):
    """A lattice of lo to hi sites: (kind, L, sites)."""
    n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    if rng.random() < 0.3:
        L = max(3, int(round(math.sqrt(n / 2))))
        return "honeycomb", L, 2 * L * L
    L = max(3, int(round(math.sqrt(n))))
    return "square", L, L * L


def draw(rng):
    """One more case of these ranges."""
    kind = rng.choice(["equal_time", "sweep", "sweep", "sweep", "sweep", "batch", "serve", "build",
                       "replay", "susceptibility", "global"])
    U = rng.choice([-1.0, -1.0, 1.0]) * round(rng.uniform(0.5, 4.0), 2)
    mu = round(rng.uniform(-0.5, 0.0), 2) if U > 0 else 0.0
    safe_mult = rng.choice([5, 8, 10, 10])
    top = {"equal_time": 700, "sweep": 800, "batch": 196, "serve": 150, "build": 700, "replay": 450,
           "susceptibility": 130, "global": 260}[kind]
    lattice, L, n = _lattice(rng, 16, top)
    slices = _log_int(rng, 15, 120 if n <= 300 else 60 if n <= 600 else 30)
    more = {}
    if kind == "equal_time":
        slices = min(slices, 30)
    elif kind == "batch":
        more = {"chains": _log_int(rng, 3, 48), "mix": rng.randrange(1 << 20)}
        slices = min(slices, 80)
    elif kind == "serve":
        more = {"chains": rng.randint(2, 8), "mix": rng.randrange(1 << 20)}
        slices = min(slices, 80)
    elif kind == "replay":
        more = {"at": rng.randint(0, slices)}
    elif kind == "susceptibility":
        slices = min(slices, 60)
        more = {"observable": rng.choice(["charge", "x", "z"])}
    elif kind == "global":
        more = {"flips": rng.randint(1, 12)}
    c = _case("", kind, lattice, L, U, mu, slices, safe_mult, **more)
    del c["name"]
    return c


def _members(case):
    """The chains of a case: one, or a mix of shapes up to the case's own (given by `mix`)."""
    if "chains" not in case:
        return [case]
    r = random.Random(case["mix"])
    out = []
    for _ in range(case["chains"]):
        U = r.choice([-1.0, 1.0]) * r.uniform(0.5, abs(case["U"]))
        L = r.randint(min(4, case["L"]), case["L"]) if case["kind"] == "serve" else \
            r.choice([x for x in (3, 4, 6, 8, 10, 12, 16) if x <= case["L"]])
        out.append(dict(case, L=L, U=U, mu=case["mu"] if U > 0 else 0.0,
                        slices=max(10, r.randint(4, 10) * case["slices"] // 10)))
    return out


def _flavours(case):
    return 2 if case["U"] < 0 else 1


def _sites(case):
    return case["L"] ** 2 * (2 if case["lattice"] == "honeycomb" else 1)


def _alpha(case):
    return math.acosh(math.exp(0.5 * DTAU * abs(case["U"])))


def _field(case, rng):
    """A +-1 field as a running chain has it: random, one slice much like the next."""
    n, M = _sites(case), case["slices"]
    flips = np.where(rng.random((n, M)) < 0.3, -1, 1)
    return np.asfortranarray(np.cumprod(flips, axis=1), dtype=np.int8)


def _inputs(case, seed):
    """Per chain: (case, field, seed of the Metropolis uniforms)."""
    rng = np.random.default_rng(seed)
    return [(c, _field(c, rng), int(rng.integers(1 << 40))) for c in _members(case)]


def _proposal_mask(case, seed):
    """The +-1 factor of a global move: a few sites flipped on every slice."""
    rng = np.random.default_rng([seed, 1])
    n, M = _sites(case), case["slices"]
    mask = np.ones((n, M), dtype=np.int8, order="F")
    mask[rng.choice(n, size=min(case["flips"], n), replace=False), :] = -1
    return mask


# ---- one pass ------------------------------------------------------------------------------
def _model(case):
    pkg = _pkg()
    l = pkg.Honeycomb(case["L"]) if case["lattice"] == "honeycomb" else pkg.SquareLattice(case["L"])
    return pkg.HubbardModel(l=l, U=case["U"], mu=case["mu"])


def _chain(case, model, field, seed):
    from montecarlo_jl_amd import _lib
    ch = _lib.HIPChain(_sites(case), _flavours(case), case["slices"], case["safe_mult"], DTAU, _alpha(case))
    ch.set_hopping(model.hopping_matrix())
    ch.set_field(field)
    ch.set_seed(seed)
    ch.build_stack()
    return ch


def prepare(case, seed):
    pkg = _pkg()
    from montecarlo_jl_amd import _lib
    inputs = _inputs(case, seed)
    models = [_model(c) for c, _, _ in inputs]
    s = {"case": case, "inputs": inputs, "lattice": models[0].l}
    if case["kind"] == "serve":
        s["server"] = _lib.Server(memory_budget=32 << 30, max_active=8)
        s["requests"] = [(m.hopping_matrix(), f, _flavours(c), c["safe_mult"], DTAU, _alpha(c), u, 1)
                         for m, (c, f, u) in zip(models, inputs)]
        return s
    s["chains"] = [_chain(c, m, f, u) for m, (c, f, u) in zip(models, inputs)]
    if case["kind"] == "global":
        s["mask"] = _proposal_mask(case, seed)
    return s


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "serve":
        srv = s["server"]
        ids = [srv.submit(*r) for r in s["requests"]]
        for i in ids:
            srv.wait(i)
        got = [srv.result(i) for i in ids]
        return [{k: r[k] for k in ("field", "greens", "accepted")} for r in got]
    if kind == "batch":
        from montecarlo_jl_amd import _lib
        accepted = _lib.batch_sweep(s["chains"], 1)
        G = [c.greens().ravel() for c in s["chains"]]
        fields = [c.get_field().ravel() for c in s["chains"]]
        # in groups of eight chains
        return {"accepted": accepted, "field": np.concatenate(fields),
                "greens": [np.concatenate(G[i:i + 8]) for i in range(0, len(G), 8)]}
    ch = s["chains"][0]
    if kind == "sweep":
        accepted = ch.sweep(1)
        return {"accepted": accepted, "field": ch.get_field(), "greens": ch.greens(physical=True)}
    if kind == "equal_time":
        return ch.measure_equal_time(case["U"])
    if kind == "build":
        ch.set_field(s["inputs"][0][1])
        ch.build_stack()
        return ch.greens()
    if kind == "replay":
        ch.set_field(s["inputs"][0][1])
        return ch.calculate_greens(case["at"])
    if kind == "susceptibility":
        accepted = ch.sweep(1)
        chi = ch.density_susceptibility(s["lattice"], case["observable"], recalculate=case["safe_mult"])
        return {"accepted": accepted, "field": ch.get_field(), "chi": chi}
    if kind == "global":
        accepted, p = ch.global_update(ch.get_field() * s["mask"])
        return {"accepted": accepted, "p": p, "field": ch.get_field(), "greens": ch.greens()}
    raise ValueError(kind)


# ---- the work a pass cannot do without --------------------------------------------------------
def _sweep_work(c):
    """Per flavour block: 2M wraps and M chunk products each way (12 M n^3), 2K stabilisations of
    two decompositions and a solve (46 K n^3), and the rank-1 updates of half the proposals."""
    n, M, b = _sites(c), c["slices"], _flavours(c)
    K = -(-M // c["safe_mult"])
    return b * (n ** 3 * (12.0 * M + 46.0 * K) + 2.0 * n * n * n * M)


def _build_work(c, chunks=None):
    """Chunk products, a decomposition with its product per chunk, and one G."""
    n, M, b = _sites(c), c["slices"], _flavours(c)
    K = -(-M // c["safe_mult"])
    return b * n ** 3 * (2.0 * M + 6.0 * K + 15.0)


def work(case):
    by, fl = 0.0, 0.0
    for c in _members(case):
        n, M, b = _sites(c), c["slices"], _flavours(c)
        io = 8.0 * b * n * n
        kind = case["kind"]
        if kind == "equal_time":
            by += io + 8.0 * n * n + 8.0 * (5 + (b + 1) * n)
            fl += 2.0 * b * n * n + 4.0 * b * n ** 3
            continue
        by += 2.0 * n * M + io
        if kind in ("sweep", "batch"):
            fl += _sweep_work(c)
        elif kind == "serve":
            fl += _sweep_work(c) + _build_work(c)
            by += 8.0 * n * n
        elif kind in ("build", "replay", "global"):
            fl += _build_work(c)
        else:
            K = -(-M // c["safe_mult"])
            # per slice three products each to advance and to transform the triple, per chunk
            # three Green's functions (three decompositions and two solves each)
            fl += _sweep_work(c) + b * n ** 3 * (18.0 * M + 3 * 25.0 * K)
    return {"bytes": by, "flops": fl}


# ---- the same results in plain numpy ------------------------------------------------------------
def _hopping(c):
    """Nearest-neighbour hopping on a periodic lattice, site = cell + cells * basis."""
    L, n = c["L"], _sites(c)
    T = np.zeros((n, n))
    cell = lambda x, y: (x % L) + L * (y % L)
    for x in range(L):
        for y in range(L):
            i = cell(x, y)
            if c["lattice"] == "honeycomb":
                for j in (cell(x, y), cell(x - 1, y), cell(x, y - 1)):
                    T[i, L * L + j] -= 1.0
                    T[L * L + j, i] -= 1.0
            else:
                for j in (cell(x + 1, y), cell(x, y + 1), cell(x - 1, y), cell(x, y - 1)):
                    T[j, i] -= 1.0
    T[np.arange(n), np.arange(n)] -= c["mu"]
    return T


def _uniform(seed, k):
    m = (1 << 64) - 1
    z = (seed + (k + 1) * 0x9E3779B97F4A7C15) & m
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & m
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & m
    return ((z ^ (z >> 31)) >> 11) * 2.0 ** -53


def _graded(A):
    """A = U diag(D) T from a QR of the columns in the order of their norms."""
    order = np.argsort(-np.linalg.norm(A, axis=0), kind="stable")
    Q, R = np.linalg.qr(A[:, order])
    D = np.abs(np.diag(R))
    T = np.empty_like(A)
    T[:, order] = R / D[:, None]
    return Q, D, T


def _inverse(l, r):
    """(I + Ul Dl Tl (Ur Dr Tr)^T)^-1 and log |det| of its inverse, large and small scales kept apart."""
    (Ul, Dl, Tl), (Ur, Dr, Tr) = l, r
    a, b = np.maximum(Dl, 1.0), np.maximum(Dr, 1.0)
    mid = (Ul.T @ Ur) / a[:, None] / b[None, :] + (Dl / a)[:, None] * (Tl @ Tr.T) * (Dr / b)[None, :]
    logdet = np.log(a).sum() + np.log(b).sum() + np.linalg.slogdet(mid)[1]
    return (Ur / b[None, :]) @ np.linalg.solve(mid, Ul.T / a[:, None]), logdet


class _Plain:
    """One chain in plain numpy: B_l = e^{-dtau T} e^{+-alpha x_l} per flavour,
    G_l = (I + B_l .. B_1 B_M .. B_{l+1})^-1."""

    def __init__(self, c, field, seed):
        self.c, self.x, self.seed, self.used = c, field.astype(np.float64), seed, 0
        self.T = _hopping(c)
        w, V = np.linalg.eigh(self.T)
        ex = lambda f: (V * np.exp(f * DTAU * w)[None, :]) @ V.T
        self.em, self.ep, self.hm, self.hp = ex(-1.0), ex(1.0), ex(-0.5), ex(0.5)
        self.b, self.M, self.n, self.a = _flavours(c), c["slices"], _sites(c), _alpha(c)
        self.chunk = 5
        self.stops = list(range(0, self.M, self.chunk)) + [self.M]

    def ev(self, f, s, power=1.0):
        return np.exp(power * (1.0 if f == 0 else -1.0) * self.a * self.x[:, s - 1])

    def unit(self):
        return np.eye(self.n), np.ones(self.n), np.eye(self.n)

    def left(self, f, udt, lo, hi):
        """B_hi .. B_{lo+1} U D T."""
        U, D, T = udt
        for s in range(lo + 1, hi + 1):
            U = self.em @ (self.ev(f, s)[:, None] * U)
        U, D, t = _graded(U * D[None, :])
        return U, D, t @ T

    def right(self, f, udt, lo, hi):
        """(B_hi .. B_{lo+1})^T U D T."""
        U, D, T = udt
        for s in range(hi, lo, -1):
            U = self.ev(f, s)[:, None] * (self.em @ U)
        U, D, t = _graded(U * D[None, :])
        return U, D, t @ T

    def green(self, f, l=0):
        """G_l from scratch and log |det(I + B_M .. B_1)|."""
        lft, rgt = self.unit(), self.unit()
        for lo in range(0, l, self.chunk):
            lft = self.left(f, lft, lo, min(lo + self.chunk, l))
        for hi in range(self.M, l, -self.chunk):
            rgt = self.right(f, rgt, max(hi - self.chunk, l), hi)
        return _inverse(lft, rgt)

    def greens(self, l=0):
        return [self.green(f, l)[0] for f in range(self.b)]

    def physical(self, G):
        return np.stack([self.hp @ g @ self.hm for g in G])

    def visit(self, G, s):
        """All sites of slice s in order, G = G_{s-1}; rank-1 updates gathered in blocks."""
        n, top = self.n, 64
        C, R = np.empty((self.b, n, top)), np.empty((self.b, top, n))
        diag = [np.diag(g).copy() for g in G]
        m, got = 0, 0
        for i in range(n):
            x = self.x[i, s - 1]
            d = [math.exp(-2.0 * self.a * x * (1.0 if f == 0 else -1.0)) - 1.0 for f in range(self.b)]
            r = [1.0 + d[f] * (1.0 - diag[f][i]) for f in range(self.b)]
            p = math.exp(2.0 * self.a * x) * r[0] * r[0] if self.b == 1 else r[0] * r[1]
            if not p > 1.0:
                self.used += 1
                if not _uniform(self.seed, self.used - 1) < p:
                    continue
            for f in range(self.b):
                u = -(G[f][:, i] - C[f][:, :m] @ R[f][:m, i])
                v = (d[f] / r[f]) * (G[f][i, :] - C[f][i, :m] @ R[f][:m, :])
                u[i] += 1.0
                C[f][:, m], R[f][m] = u, v
                diag[f] -= u * v
            self.x[i, s - 1] = -x
            got, m = got + 1, m + 1
            if m == top:
                for f in range(self.b):
                    G[f] -= C[f] @ R[f]
                m = 0
        for f in range(self.b):
            G[f] -= C[f][:, :m] @ R[f][:m]
        return got

    def sweep(self):
        """Slices 1 .. M, then M .. 1, G from the decompositions at every chunk's end."""
        got, K, st = 0, len(self.stops) - 1, self.stops
        rgt = [[self.unit()] for _ in range(self.b)]
        for k in range(K - 1, -1, -1):
            for f in range(self.b):
                rgt[f].append(self.right(f, rgt[f][-1], st[k], st[k + 1]))
        lft = [[self.unit()] for _ in range(self.b)]
        for k in range(K):
            G = [_inverse(lft[f][k], rgt[f][K - k])[0] for f in range(self.b)]
            for s in range(st[k] + 1, st[k + 1] + 1):
                got += self.visit(G, s)
                for f in range(self.b):
                    G[f] = (self.em @ (self.ev(f, s)[:, None] * G[f] * self.ev(f, s, -1.0)[None, :])) @ self.ep
            for f in range(self.b):
                lft[f].append(self.left(f, lft[f][k], st[k], st[k + 1]))
        rgt = [self.unit() for _ in range(self.b)]
        for k in range(K - 1, -1, -1):
            G = [_inverse(lft[f][k + 1], rgt[f])[0] for f in range(self.b)]
            for s in range(st[k + 1], st[k], -1):
                for f in range(self.b):
                    G[f] = self.ev(f, s, -1.0)[:, None] * (self.ep @ G[f] @ self.em) * self.ev(f, s)[None, :]
                got += self.visit(G, s)
            rgt = [self.right(f, rgt[f], st[k], st[k + 1]) for f in range(self.b)]
        return got

    def displaced(self, f):
        """(G(0, l), G(l, 0), G(l, l)) for l = 0 .. M from the inverse of the block cyclic matrix of
        short slice products."""
        n, M, step = self.n, self.M, 3
        B = [self.em * self.ev(f, s)[None, :] for s in range(1, M + 1)]
        Bi = [self.ev(f, s, -1.0)[:, None] * self.ep for s in range(1, M + 1)]
        at = list(range(0, M, step))
        K = len(at)
        O = np.eye(n * K)
        for k in range(K):
            P = np.eye(n)
            for s in range(at[k], at[k + 1] if k + 1 < K else M):
                P = B[s] @ P
            j = (k + 1) % K
            O[j * n:(j + 1) * n, k * n:(k + 1) * n] += P if j == 0 else -P
        g = np.linalg.inv(O)
        blk = lambda k, l: g[k * n:(k + 1) * n, l * n:(l + 1) * n]
        out = []
        for k in range(K):
            G0l, Gl0, Gll = blk(0, k), blk(k, 0), blk(k, k)
            out.append((G0l, Gl0, Gll))
            for s in range(at[k], (at[k + 1] if k + 1 < K else M + 1) - 1):
                if k == 0 and s == 0:
                    G0l = G0l - np.eye(n)     # past equal times: -(I - G) on this side
                G0l, Gl0, Gll = G0l @ Bi[s], B[s] @ Gl0, B[s] @ Gll @ Bi[s]
                out.append((G0l, Gl0, Gll))
        return out

    def susceptibility(self, observable):
        """(1/N) int dtau sum_src <O_i(tau) O_j(0)> by distance, the full kernels, G00 = the chain's G."""
        c, n, M, b, L = self.c, self.n, self.M, self.b, self.c["L"]
        cells = L * L
        basis = n // cells
        xs, ys = np.arange(cells) % L, np.arange(cells) // L
        trip = [[tuple(self.hp @ X @ self.hm for X in t) for t in self.displaced(f)] for f in range(b)]
        G00 = [t[0][0] for t in trip]
        out = np.zeros((cells, basis, basis))
        src = np.arange(cells)
        for l in range(M + 1):
            w = DTAU * (0.5 if l in (0, M) else 1.0)
            for d in range(cells):
                trg = (xs + xs[d]) % L + L * ((ys + ys[d]) % L)
                for b1 in range(basis):
                    for b2 in range(basis):
                        i, j = src + b1 * cells, trg + b2 * cells
                        one = ((i == j) & (l == 0)).astype(float)
                        con = lambda f, h: (one - trip[f][l][0][j, i]) * trip[h][l][1][i, j]
                        oi = [1.0 - trip[f][l][2][i, i] for f in range(b)]
                        oj = [1.0 - G00[f][j, j] for f in range(b)]
                        if b == 1:
                            v = 2.0 * con(0, 0) + (4.0 * oi[0] * oj[0] if observable == "charge" else 0.0)
                        elif observable == "charge":
                            v = (oi[0] + oi[1]) * (oj[0] + oj[1]) + con(0, 0) + con(1, 1)
                        elif observable == "z":
                            v = (oi[0] - oi[1]) * (oj[0] - oj[1]) + con(0, 0) + con(1, 1)
                        else:
                            v = con(0, 1) + con(1, 0)
                        out[d, b1, b2] += w * v.sum()
        return out / n


def _equal_time(p, U):
    G = p.physical(p.greens())
    kin = sum(float(np.sum(p.T * (np.eye(p.n) - g))) for g in G) * (2.0 if p.b == 1 else 1.0)
    up, dn = np.diag(G[0]), np.diag(G[-1])
    inter = -U * float(np.sum((up - 0.5) * (dn - 0.5)))
    docc = (1.0 - up) * (1.0 - dn)
    return {"density": float(np.mean(2.0 - up - dn)), "kinetic_energy": kin, "interaction_energy": inter,
            "total_energy": kin + inter, "mean_double_occupancy": float(docc.mean()),
            "occupation": np.concatenate([1.0 - np.diag(g) for g in G]), "double_occupancy": docc}


def exact(case, seed):
    kind = case["kind"]
    inputs = _inputs(case, seed)
    if kind in ("batch", "serve"):
        got = []
        for c, f, u in inputs[:8]:
            p = _Plain(c, f, u)
            got.append((p.sweep(), np.stack(p.greens())))
        if kind == "serve":
            return [{"field": None, "greens": G, "accepted": a} for a, G in got]
        groups = [np.concatenate([G.ravel() for _, G in got])]
        return {"accepted": None, "field": None, "greens": groups + [None] * (-(-len(inputs) // 8) - 1)}
    if _sites(case) > 600 and kind == "sweep":
        return None
    p = _Plain(*inputs[0])
    if kind == "sweep":
        a = p.sweep()
        return {"accepted": a, "field": None, "greens": p.physical(p.greens())}
    if kind == "equal_time":
        return _equal_time(p, case["U"])
    if kind == "build":
        return np.stack(p.greens())
    if kind == "replay":
        return np.stack(p.greens(case["at"]))
    if kind == "susceptibility":
        a = p.sweep()
        if _sites(case) * case["slices"] > 9000:
            return {"accepted": a, "field": None, "chi": None}
        return {"accepted": a, "field": None, "chi": p.susceptibility(case["observable"])}
    # a global update: the ratio of the weights, one uniform where it is not above 1
    q = _Plain(inputs[0][0], inputs[0][1] * _proposal_mask(case, seed), inputs[0][2])
    old, new = ([x.green(f) for f in range(x.b)] for x in (p, q))
    log = sum(b[1] - a[1] for a, b in zip(old, new)) * (2.0 if p.b == 1 else 1.0)
    if p.b == 1:
        log -= p.a * float(q.x.sum() - p.x.sum())
    ratio = math.exp(log)
    accepted = ratio > 1.0 or _uniform(inputs[0][2], 0) < ratio
    return {"accepted": accepted, "p": ratio, "field": None,
            "greens": np.stack([g[0] for g in (new if accepted else old)])}
