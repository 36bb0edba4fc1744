"""The work this library is timed on: what a quantum-chemistry program has it do.

Per geometry a program uploads the basis, computes the Schwarz bounds and keeps
the handle with its work lists; per SCF cycle it asks for the two-electron
operator G(D) (HF, or B3LYP's exchange weight 0.2) and, for B3LYP, V_xc; per
geometry step for the one-electron integrals and for the four-centre gradient.
The basis is 6-31G** throughout.  Systems are seeded water clusters and
n-alkanes, from one molecule to (H2O)64; densities decay with distance as a
converged one does.  The geometry and the density come from the seed, so
another seed is another molecule of the same kind.
"""
from __future__ import annotations

import itertools
import math

import numpy as np
import torch

from quick_amd.basis import build_basis
from quick_amd.fock import QK_FP64, QK_MIXED, FockEngine, make_opts
from quick_amd.geometry import n_alkane, synthetic_density, water_cluster
from quick_amd.xc import QK_GRID_PRODUCT, QK_GRID_SG1, XcEngine, make_xc_opts


def _water(nx, ny, nz):
    return {"system": "water", "nx": nx, "ny": ny, "nz": nz}


def _alkane(n):
    return {"system": "alkane", "carbons": n}


def listed():
    return [
        # one molecule: the smallest call, where launches and serial chains count
        {"name": "fock_water1", "op": "fock", **_water(1, 1, 1), "precision": "fp64", "hybrid": 1.0, "host": False},
        # a mid-sized molecule through the host-array boundary (density up, operator down)
        {"name": "fock_nonane_host", "op": "fock", **_alkane(9), "precision": "fp64", "hybrid": 1.0, "host": True},
        # the benchmark cluster in full precision: one SCF cycle's operator
        {"name": "fock_water32", "op": "fock", **_water(4, 4, 2), "precision": "fp64", "hybrid": 1.0, "host": False},
        # the same in mixed precision at the benchmark's threshold
        {"name": "fock_water32_mixed", "op": "fock", **_water(4, 4, 2), "precision": "mixed", "threshold": 1e-3,
         "hybrid": 1.0, "host": False},
        # the largest configuration: (H2O)64, 1,600 functions, B3LYP's exchange weight
        {"name": "fock_water64_b3lyp", "op": "fock", **_water(4, 4, 4), "precision": "mixed", "threshold": 1e-3,
         "hybrid": 0.2, "host": False},
        # gradient of one molecule: the smallest backward call
        {"name": "grad_water1", "op": "grad", **_water(1, 1, 1), "precision": "fp64", "hybrid": 1.0, "host": False},
        # the gradient benchmark's chain molecule, full precision
        {"name": "grad_icosane", "op": "grad", **_alkane(20), "precision": "fp64", "hybrid": 1.0, "host": False},
        # the benchmark cluster's gradient in mixed precision, with the options object of its operator builds (at a
        # threshold of 1e-2 the FP32 integrals alone put 3e-9 of the gradient's norm on it, at 1e-3 1e-10)
        {"name": "grad_water32_mixed", "op": "grad", **_water(4, 4, 2), "precision": "mixed", "threshold": 1e-3,
         "hybrid": 1.0, "host": False},
        # one-electron integrals and their gradient terms, once per geometry step
        {"name": "oneint_water32", "op": "oneint", **_water(4, 4, 2)},
        # B3LYP exchange-correlation on a caller's grid, a small cluster
        {"name": "xc_water4_grid", "op": "xc", **_water(2, 2, 1), "grid": "caller", "nrad": 40, "nang": 128},
        # B3LYP exchange-correlation of (H2O)64 on the 75 x 302 grid
        {"name": "xc_water64", "op": "xc", **_water(4, 4, 4), "grid": "product", "nrad": 75, "nang": 302},
        # a whole calculation: RHF from the core guess to convergence
        {"name": "scf_water4", "op": "scf", **_water(2, 2, 1), "precision": "fp64"},
    ]


def draw(rng):
    op = rng.choice(["fock", "fock", "fock", "grad", "grad", "oneint", "xc", "scf"])
    big = {"fock": 40, "grad": 24, "oneint": 32, "xc": 32, "scf": 4}[op]
    want = math.exp(rng.uniform(0.0, math.log(big)))
    if op != "scf" and rng.random() < 0.35:   # one carbon weighs like one water
        system = _alkane(max(2, min(20, round(want))))
    else:
        dims = [d for d in itertools.product(range(1, 5), repeat=3) if math.prod(d) <= big]
        near = min(abs(math.log(math.prod(d) / want)) for d in dims)
        system = _water(*rng.choice([d for d in dims if abs(math.log(math.prod(d) / want)) <= near + 1e-9]))
    case = {"op": op, **system}
    if op in ("fock", "grad"):
        case["hybrid"] = rng.choice([1.0, 1.0, 0.2])
        case["precision"] = rng.choice(["fp64", "mixed"])
        if case["precision"] == "mixed":
            case["threshold"] = math.exp(rng.uniform(math.log(1e-5), math.log(1e-3)))
        case["host"] = rng.random() < 0.3
    elif op == "scf":
        case["precision"] = "fp64"
    elif op == "xc":
        case["grid"] = rng.choice(["caller", "sg1", "product"])
        if case["grid"] == "caller":
            case["nrad"], case["nang"] = rng.randrange(20, 60), rng.choice([50, 72, 128, 162])
        if case["grid"] == "product":
            case["nrad"], case["nang"] = rng.randrange(30, 76), rng.choice([86, 194, 302])
    return case


# ---------------------------------------------------------------- inputs

def _basis(case, seed):
    if case["system"] == "water":
        s, x = water_cluster(case["nx"], case["ny"], case["nz"], seed=seed)
    else:
        s, x = n_alkane(case["carbons"], seed=seed)
    return build_basis(s, x)


def _density(b, seed):
    return synthetic_density(b.xyz, b.katom, b.ksumtype, b.nbasis, seed + 1)


def _positive_density(b, seed):
    """a density of occupied orbitals (rho >= 0 everywhere) with the electron count of the molecule, about"""
    u = np.random.default_rng(seed + 1).uniform(-1.0, 1.0, (b.nbasis, max(1, b.nelec // 2)))
    at = _centres(b)
    home = np.sort(np.random.default_rng(seed + 2).integers(0, b.natom, u.shape[1]))
    r2 = ((b.xyz[:, at].T[:, None, :] - b.xyz[:, home].T[None, :, :]) ** 2).sum(-1)
    c = u * np.exp(-0.125 * r2)
    return (b.nelec / float((c * c).sum())) * (c @ c.T)


def _centres(b):
    at = np.zeros(b.nbasis, np.int64)
    for s in range(b.nshell):
        at[b.ksumtype[s] - 1:b.ksumtype[s + 1] - 1] = b.katom[s] - 1
    return at


def _grid(b, nrad, nang):
    """(x, y, z, w) rows: Becke-partitioned atomic grids, Gauss-Chebyshev radii times a Gauss-Legendre x trapezoid
    sphere of about nang points"""
    nth = max(2, round(math.sqrt(nang / 2)))
    nph = max(3, nang // nth)
    ct, wt = np.polynomial.legendre.leggauss(nth)
    ph = 2 * math.pi * (np.arange(nph) + 0.5) / nph
    st = np.sqrt(1 - ct ** 2)
    u = np.stack([np.outer(st, np.cos(ph)), np.outer(st, np.sin(ph)), np.outer(ct, np.ones(nph))], -1).reshape(-1, 3)
    wu = np.repeat(wt * 2 * math.pi / nph, nph)
    i = np.arange(1, nrad + 1)
    x = np.cos(i * math.pi / (nrad + 1))
    r = (1 + x) / (1 - x)
    wr = math.pi / (nrad + 1) * np.sin(i * math.pi / (nrad + 1)) * 2 / (1 - x) ** 2 * r ** 2
    keep = r < 20.0
    r, wr = r[keep], wr[keep]
    A = b.xyz.T
    dist = np.linalg.norm(A[:, None] - A[None], axis=-1) + np.eye(len(A))
    rows = []
    for a in range(len(A)):
        p = (A[a] + r[:, None, None] * u[None]).reshape(-1, 3)
        w = (wr[:, None] * wu[None]).reshape(-1)
        d = np.linalg.norm(p[:, None] - A[None], axis=-1)
        cell = np.ones_like(d)
        for k in range(len(A)):
            mu = (d[:, k:k + 1] - d) / dist[k]
            for _ in range(3):
                mu = 1.5 * mu - 0.5 * mu ** 3
            s = 0.5 * (1 - mu)
            s[:, k] = 1.0
            cell[:, k] = s.prod(1)
        rows.append(np.column_stack([p, w * cell[:, a] / cell.sum(1)]))
    g = np.concatenate(rows)
    return g[g[:, 3] > 1e-10]


def _opts(case):
    if case["precision"] == "mixed":
        return make_opts(hybrid=case["hybrid"], precision=QK_MIXED, fp32_threshold=case["threshold"])
    return make_opts(hybrid=case["hybrid"], precision=QK_FP64)


def _fortran(a):
    return np.asfortranarray(a).ravel(order="F").copy()


def prepare(case, seed):
    b = _basis(case, seed)
    st = {"case": case, "stream": torch.cuda.current_stream().cuda_stream}
    if case["op"] == "xc":
        eng = XcEngine(b)
        if case["grid"] == "caller":
            eng.set_grid(_grid(b, case["nrad"], case["nang"]))
        elif case["grid"] == "sg1":
            eng.build_grid(make_xc_opts(grid=QK_GRID_SG1))
        else:
            eng.build_grid(make_xc_opts(grid=QK_GRID_PRODUCT, nrad=case["nrad"], nang=case["nang"]))
        D = torch.from_numpy(_fortran(_positive_density(b, seed))).cuda()
        return {**st, "engine": eng, "D": D, "V": torch.empty_like(D)}
    eng = FockEngine(b)
    eng.compute_schwarz()
    if case["op"] in ("oneint", "scf"):
        eng.set_charges(b.Z.astype(float))
    if case["op"] == "oneint":
        return {**st, "engine": eng, "D": _density(b, seed), "W": _density(b, seed + 10)}
    if case["op"] == "scf":
        return {**st, "engine": eng, "nocc": b.nelec // 2}
    o = _opts(case)
    eng.prepare(o)
    D = _density(b, seed)
    st |= {"engine": eng, "opts": o}
    if case["host"]:
        return {**st, "D": D}
    D = torch.from_numpy(_fortran(D)).cuda()
    if case["op"] == "fock":
        return {**st, "D": D, "out": torch.empty_like(D)}
    return {**st, "D": D, "out": torch.zeros(3 * b.natom, dtype=torch.float64, device="cuda")}


def run(st):
    case, eng = st["case"], st["engine"]
    if case["op"] == "fock":
        if case["host"]:
            return eng.fock(st["D"], st["opts"])
        eng.fock_device(st["D"].data_ptr(), st["out"].data_ptr(), st["opts"], st["stream"])
        return st["out"]
    if case["op"] == "grad":
        if case["host"]:
            return eng.grad(st["D"], st["opts"])
        st["out"].zero_()
        eng.grad_device(st["D"].data_ptr(), st["out"].data_ptr(), st["opts"], st["stream"])
        return st["out"]
    if case["op"] == "oneint":
        S, H = eng.oneint()
        return {"S": S, "H": H, "grad": eng.oneint_grad(st["D"], st["W"])}
    if case["op"] == "xc":
        E, N = eng.xc_device(st["D"].data_ptr(), st["V"].data_ptr(), st["stream"])
        return {"V": st["V"], "Exc": E, "electrons": N}
    D, E, _, _ = eng.scf(st["nocc"])
    return {"D": D, "E": E}


def _size(case):
    """(units of one water or one carbon, functions, atoms)"""
    if case["system"] == "water":
        m = case["nx"] * case["ny"] * case["nz"]
        return m, 25 * m, 3 * m
    c = case["carbons"]
    return c, 15 * c + 5 * (2 * c + 2), 3 * c + 2


def work(case):
    """The arithmetic of the surviving integrals, by the library's own per-class operation counts, fitted over the
    cluster and chain sizes at these cutoffs and densities; the bytes are the density, the result and the
    primitive-pair data (56 bytes each) read or written once."""
    m, n, natom = _size(case)
    near = min(m, 12)
    prims = 230 * m * near
    if case["op"] in ("fock", "grad", "scf"):
        a, c, d = FOCK_FLOPS[case["system"]]
        flops = math.exp(a + c * math.log(m) + d * math.log(m) ** 2)
        if case["op"] == "grad":
            return {"bytes": 8 * n * n + 24 * natom + 56 * prims, "flops": 5 * flops}
        if case["op"] == "scf":   # about 20 cycles, each an operator and some ten n^3 products
            return {"bytes": 20 * (16 * n * n + 56 * prims), "flops": 20 * (flops + 20 * n ** 3)}
        return {"bytes": 16 * n * n + 56 * prims, "flops": flops}
    if case["op"] == "oneint":
        # per primitive pair and nucleus one Boys function and a few dozen integrals, and the same for three gradients
        return {"bytes": 32 * n * n + 56 * prims, "flops": 4 * 300.0 * prims * natom}
    pts = {"caller": case.get("nrad", 0) * case.get("nang", 0) * 0.8, "sg1": 3300.0,
           "product": case.get("nrad", 0) * case.get("nang", 0) * 0.67}[case["grid"]] * natom
    near = min(n, 160)   # functions that reach a point
    return {"bytes": 16 * n * n + 32 * pts, "flops": pts * (4.0 * near * near + 80 * near + 500)}


#: ln(flops) of one operator as a polynomial in ln(units): fitted from one to 64 waters, two to 20 carbons
FOCK_FLOPS = {"water": (16.04, 3.525, -0.185), "alkane": (16.77, 3.72, -0.271)}


# ---------------------------------------------------------------- 64-bit reference

class _Gauss:
    """Cartesian Gaussians as sums over primitives, by McMurchie and Davidson's Hermite expansion"""

    def __init__(self, b):
        at = _centres(b)
        prims, self.funcs = {}, []
        for s in range(b.nshell):
            f0, f1 = b.ksumtype[s] - 1, b.ksumtype[s + 1] - 1
            for f in range(f0, f1):
                lmn = tuple(int(v) for v in b.KLMN[:, f])
                col = f0 + sum(lmn)   # the shell's contraction column of this angular momentum
                terms = []
                for k in range(b.kprim[s]):
                    key = (int(at[f]), float(b.gcexpo[k, col]))
                    i = prims.setdefault(key, len(prims))
                    terms.append((i, float(b.gccoeff[k, col] * b.cons[f]), lmn))
                self.funcs.append(terms)
        self.at = at
        self.atom = np.array([k[0] for k in prims])
        self.a = np.array([k[1] for k in prims])
        self.A = np.ascontiguousarray(b.xyz.T[self.atom])
        n = len(self.a)
        self.ij = [(i, j) for i in range(n) for j in range(i, n)]
        self.where = {p: k for k, p in enumerate(self.ij)}
        I, J = np.array(self.ij).T
        self.p = self.a[I] + self.a[J]
        self.P = (self.a[I, None] * self.A[I] + self.a[J, None] * self.A[J]) / self.p[:, None]
        self.E = [self._e1d(I, J, x) for x in range(3)]

    def _e1d(self, I, J, x, lmax=4):
        """E[l1][l2][t] per primitive pair, one direction"""
        p, mu = self.p, self.a[I] * self.a[J] / self.p
        d = self.A[I, x] - self.A[J, x]
        pa, pb = self.P[:, x] - self.A[I, x], self.P[:, x] - self.A[J, x]
        E = {(0, 0, 0): np.exp(-mu * d * d)}
        get = lambda i, j, t: E.get((i, j, t), 0.0)
        for s in range(1, 2 * lmax + 1):
            for i in range(max(0, s - lmax), min(lmax, s) + 1):
                j = s - i
                for t in range(s + 1):
                    if i > 0:
                        E[i, j, t] = get(i - 1, j, t - 1) / (2 * p) + pa * get(i - 1, j, t) + (t + 1) * get(i - 1, j, t + 1)
                    else:
                        E[i, j, t] = get(i, j - 1, t - 1) / (2 * p) + pb * get(i, j - 1, t) + (t + 1) * get(i, j - 1, t + 1)
        return E

    def moved(self, f, x):
        """d/d(centre) of a function, direction x"""
        out = []
        for i, c, l in f:
            up = tuple(v + (k == x) for k, v in enumerate(l))
            out.append((i, 2 * self.a[i] * c, up))
            if l[x]:
                out.append((i, -l[x] * c, tuple(v - (k == x) for k, v in enumerate(l))))
        return out

    def laplace(self, f):
        """-1/2 the Laplacian of a function"""
        out = []
        for i, c, l in f:
            for x in range(3):
                a = self.a[i]
                out.append((i, -0.5 * c * 4 * a * a, tuple(v + 2 * (k == x) for k, v in enumerate(l))))
                out.append((i, 0.5 * c * 2 * a * (2 * l[x] + 1), l))
                if l[x] > 1:
                    out.append((i, -0.5 * c * l[x] * (l[x] - 1), tuple(v - 2 * (k == x) for k, v in enumerate(l))))
        return out

    def rows(self, pairs, L):
        """Hermite coefficients of the products of pairs: (pairs, primitive pairs * tuvs(L))"""
        T = {t: k for k, t in enumerate(tuvs(L))}
        H = np.zeros((len(pairs), len(self.ij), len(T)))
        for r, (f, g) in enumerate(pairs):
            groups = {}
            for i, c, l in f:
                for j, d, m in g:
                    key = (l, m, i <= j)
                    groups.setdefault(key, []).append((self.where[(min(i, j), max(i, j))], c * d))
            for (l, m, straight), items in groups.items():
                k = np.array([v[0] for v in items])
                c = np.array([v[1] for v in items])
                u, v = (l, m) if straight else (m, l)
                ex = [[self.E[x][u[x], v[x], t][k] for t in range(u[x] + v[x] + 1)] for x in range(3)]
                for tx, ty, tz in itertools.product(*(range(len(e)) for e in ex)):
                    np.add.at(H[r, :, T[tx, ty, tz]], k, c * ex[0][tx] * ex[1][ty] * ex[2][tz])
        return H


def tuvs(L):
    return [(t, u, v) for s in range(L + 1) for t in range(s, -1, -1) for u in range(s - t, -1, -1) for v in [s - t - u]]


def _boys(m, T):
    """F_0 .. F_m: the ascending series below T = 40 for F_m, downward recursion; the asymptotic form above"""
    T = np.asarray(T, np.float64)
    F = np.zeros((m + 1,) + T.shape)
    lo = T < 40.0
    t = T[lo]
    term = np.full_like(t, 1.0 / (2 * m + 1))
    s = term.copy()
    for k in range(1, 200):
        term = term * (2 * t) / (2 * m + 2 * k + 1)
        s += term
        if not term.size or float(term.max()) < 1e-18:
            break
    e = np.exp(-t)
    f = e * s
    F[m][lo] = f
    for k in range(m - 1, -1, -1):
        f = (2 * t * f + e) / (2 * k + 1)
        F[k][lo] = f
    h = T[~lo]
    f = 0.5 * np.sqrt(math.pi / h)
    F[0][~lo] = f
    for k in range(1, m + 1):
        f = f * (2 * k - 1) / (2 * h) - np.exp(-h) / (2 * h)
        F[k][~lo] = f
    return F


def _hermite_r(alpha, R, L):
    """R_tuv for |tuv| <= L; alpha and R (.., 3) broadcast"""
    F = _boys(L, alpha * (R * R).sum(-1))
    cur = {(0, 0, 0): [(-2 * alpha) ** n * F[n] for n in range(L + 1)]}
    for t, u, v in tuvs(L)[1:]:
        s = (t, u, v)
        x = next(k for k in range(3) if s[k])
        one = tuple(c - (k == x) for k, c in enumerate(s))
        two = tuple(c - 2 * (k == x) for k, c in enumerate(s))
        out = []
        for n in range(L - sum(s) + 1):
            val = R[..., x] * cur[one][n + 1]
            if s[x] > 1:
                val = val + (s[x] - 1) * cur[two][n + 1]
            out.append(val)
        cur[s] = out
    return {s: v[0] for s, v in cur.items()}


def _eri(g, left, right, Ll, Lr):
    """(left | right) for Hermite rows of both"""
    tl, tr = tuvs(Ll), tuvs(Lr)
    sign = np.array([(-1.0) ** sum(t) for t in tr])
    n = len(g.ij)
    out = np.zeros((left.shape[0], right.shape[0]))
    Rr = (right * sign).reshape(right.shape[0], -1)
    step = 24
    for k in range(0, n, step):
        p = g.p[k:k + step]
        al = p[:, None] * g.p[None] / (p[:, None] + g.p[None])
        R = _hermite_r(al, g.P[k:k + step, None] - g.P[None], Ll + Lr)
        pre = 2 * math.pi ** 2.5 / (p[:, None] * g.p[None] * np.sqrt(p[:, None] + g.p[None]))
        M = np.empty((len(p), len(tl), n, len(tr)))
        for a, s in enumerate(tl):
            for c, t in enumerate(tr):
                M[:, a, :, c] = pre * R[tuple(i + j for i, j in zip(s, t))]
        out += left[:, k:k + step].reshape(left.shape[0], -1) @ (M.reshape(len(p) * len(tl), -1) @ Rr.T)
    return out


def _exact_two(case, seed, b):
    g = _Gauss(b)
    n, h, D = b.nbasis, case["hybrid"], _density(b, seed)
    iu = [(i, j) for i in range(n) for j in range(i, n)]
    ket = g.rows([(g.funcs[i], g.funcs[j]) for i, j in iu], 4)
    full = np.zeros((n, n), np.int64)
    for k, (i, j) in enumerate(iu):
        full[i, j] = full[j, i] = k
    if case["op"] == "fock":
        I = _eri(g, ket, ket, 4, 4)[full][:, :, full]
        G = np.einsum("abcd,cd->ab", I, D) - 0.5 * h * np.einsum("acbd,cd->ab", I, D)
        return G if case["host"] else _fortran(G)
    grad = np.zeros((3, b.natom))
    for x in range(3):
        bra = g.rows([(g.moved(g.funcs[i], x), g.funcs[j]) for i in range(n) for j in range(n)], 5)
        I = _eri(g, bra, ket, 5, 4)[:, full].reshape(n, n, n, n)
        J = np.einsum("abcd,cd->ab", I, D)
        K = np.einsum("abcd,bd->ac", I, D)
        per = 2 * (D * J).sum(1) - h * (D * K).sum(1)
        np.add.at(grad[x], g.at, per)
    return grad if case["host"] else _fortran(grad)


def _exact_oneint(case, seed, b):
    g = _Gauss(b)
    n, D, W = b.nbasis, _density(b, seed), _density(b, seed + 10)
    C, Z = b.xyz.T, b.Z.astype(float)
    R = {L: [_hermite_r(g.p, g.P - c, L + 1) for c in C] for L in (4, 5)}

    def attract(H, L, which=None, x=None):
        """sum over nuclei (or one nucleus' derivative) of the attraction of Hermite rows"""
        v = np.zeros(H.shape[0])
        for k in range(len(Z)) if which is None else [which]:
            for c, t in enumerate(tuvs(L)):
                s = t if x is None else tuple(u + (i == x) for i, u in enumerate(t))
                v += (Z[k] if x is not None else -Z[k]) * H[:, :, c] @ (2 * math.pi / g.p * R[L][k][s])
        return v

    pairs = [(i, j) for i in range(n) for j in range(n)]
    over = lambda H: H[:, :, 0] @ (math.pi / g.p) ** 1.5
    kin = lambda bra: over(g.rows([(bra(i), g.laplace(g.funcs[j])) for i, j in pairs], 7))
    H4 = g.rows([(g.funcs[i], g.funcs[j]) for i, j in pairs], 4)
    S = over(H4).reshape(n, n)
    H = (kin(lambda i: g.funcs[i]) + attract(H4, 4)).reshape(n, n)
    grad = np.zeros((3, b.natom))
    for x in range(3):
        H5 = g.rows([(g.moved(g.funcs[i], x), g.funcs[j]) for i, j in pairs], 5)
        dS = over(H5).reshape(n, n)
        dH = (kin(lambda i: g.moved(g.funcs[i], x)) + attract(H5, 5)).reshape(n, n)
        np.add.at(grad[x], g.at, 2 * (D * dH).sum(1) - 2 * (W * dS).sum(1))
        for k in range(b.natom):
            grad[x, k] += float((D.ravel() * attract(H4, 4, k, x)).sum())
            for l in range(b.natom):
                if l != k:
                    r = C[k] - C[l]
                    grad[x, k] -= Z[k] * Z[l] * r[x] / float(r @ r) ** 1.5
    return {"S": S, "H": H, "grad": grad}


def _b3lyp(rho, sigma):
    """energy per volume of the closed-shell B3LYP functional (Slater, Becke 88, VWN in RPA form, LYP)"""
    pi = math.pi
    lda = -0.75 * (3 / pi) ** (1 / 3) * rho ** (4 / 3)
    rs = rho / 2
    x = torch.sqrt(sigma) / 2 / rs ** (4 / 3)
    b88 = -2 * 0.0042 * rs ** (4 / 3) * x ** 2 / (1 + 6 * 0.0042 * x * torch.asinh(x))
    A, x0, bv, cv = 0.0310907, -0.409286, 13.072, 42.7198
    y = (3 / (4 * pi * rho)) ** (1 / 6)
    X = lambda t: t * t + bv * t + cv
    Q = math.sqrt(4 * cv - bv * bv)
    at = torch.atan(Q / (2 * y + bv))
    vwn = rho * A * (torch.log(y * y / X(y)) + 2 * bv / Q * at
                     - bv * x0 / X(x0) * (torch.log((y - x0) ** 2 / X(y)) + 2 * (bv + 2 * x0) / Q * at))
    a, b, c, d = 0.04918, 0.132, 0.2533, 0.349
    rm = rho ** (-1 / 3)
    omega = torch.exp(-c * rm) / (1 + d * rm) * rho ** (-11 / 3)
    delta = c * rm + d * rm / (1 + d * rm)
    CF = 0.3 * (3 * pi * pi) ** (2 / 3)
    saa = sigma / 4
    lyp = (-a * rho / (1 + d * rm)
           - a * b * omega * (rs * rs * (2 ** (11 / 3) * CF * 2 * rs ** (8 / 3) + (47 - 7 * delta) / 18 * sigma
                                         - (2.5 - delta / 18) * 2 * saa - (delta - 11) / 9 * saa)
                              - 2 / 3 * rho ** 2 * sigma + (2 / 3 * rho ** 2 - rs * rs) * 2 * saa))
    return 0.8 * lda + 0.72 * b88 + 0.19 * vwn + 0.81 * lyp


def _exact_xc(case, seed, b):
    grid = _grid(b, case["nrad"], case["nang"])
    D = torch.from_numpy(_positive_density(b, seed))
    at = np.asarray(b.ncenter) - 1
    V = torch.zeros(b.nbasis, b.nbasis, dtype=torch.float64)
    E = N = 0.0
    for k in range(0, len(grid), 20000):
        pts = torch.from_numpy(grid[k:k + 20000])
        phi = torch.zeros(4, len(pts), b.nbasis, dtype=torch.float64)
        for f in range(b.nbasis):
            r = pts[:, :3] - torch.from_numpy(b.xyz[:, at[f]].copy())
            nc = int(b.ncontract[f])
            al, co = torch.from_numpy(b.aexp[:nc, f].copy()), torch.from_numpy(b.dcoeff[:nc, f].copy())
            ex = co * torch.exp(-al * (r * r).sum(1, keepdim=True))
            e0, e1 = ex.sum(1), (-2 * al * ex).sum(1)
            l = [int(v) for v in b.KLMN[:, f]]
            pw = [r[:, x] ** l[x] for x in range(3)]
            poly = pw[0] * pw[1] * pw[2]
            phi[0, :, f] = poly * e0
            for x in range(3):
                dp = l[x] * r[:, x] ** max(l[x] - 1, 0) * pw[(x + 1) % 3] * pw[(x + 2) % 3]
                phi[1 + x, :, f] = dp * e0 + poly * r[:, x] * e1
        T = phi[0] @ D
        rho = (T * phi[0]).sum(1)
        gr = torch.stack([2 * (T * phi[1 + x]).sum(1) for x in range(3)], 1)
        ok = rho / 2 >= 1e-10
        phi, rho, gr, w = phi[:, ok], rho[ok].requires_grad_(), gr[ok], pts[ok, 3]
        sigma = (gr * gr).sum(1).clamp_min(1e-60).requires_grad_()
        f = _b3lyp(rho, sigma)
        vr, vs = torch.autograd.grad(f.sum(), (rho, sigma))
        z = (0.5 * w * vr)[:, None] * phi[0] + sum((2 * w * vs * gr[:, x])[:, None] * phi[1 + x] for x in range(3))
        m = phi[0].T @ z
        V += m + m.T
        E += float((w * f.detach()).sum())
        N += float((w * rho.detach()).sum())
    return {"V": _fortran(V.numpy()), "Exc": E, "electrons": N}


def exact(case, seed):
    b = _basis(case, seed)
    if case["op"] in ("fock", "grad") and b.natom <= 3:
        return _exact_two(case, seed, b)
    if case["op"] == "oneint" and b.natom <= 3:
        return _exact_oneint(case, seed, b)
    if case["op"] == "xc" and case["grid"] == "caller" and b.nbasis <= 250:
        return _exact_xc(case, seed, b)
    return None
