"""What the speed of this framework is measured on.

The cases are the work a quantum-chemistry program gives an integral library:
single quartets through the libint-style Engine, batches of quartets of the
angular momenta and contraction depths of contracted s-f basis sets, the
range-separated, mixed-precision, 3-centre and derivative variants, one-body
matrices, and screened J/K builds from a density.  Molecules are random
(minimum separation 0.9 A, 60 atoms per (14 A)^3, the density of the
repository's 60-atom workload) with the shells per atom of its recipes:
"plain" s3p2d1 with fixed depths, "spd" s4p3d2 and "spdf" s4p3d2f1 with
K ~ U{1..kmax} primitives per shell.  The exponent range narrows with l as it
does in contracted basis sets.  d and f shells are solid harmonics.

exact() evaluates the same quantities by McMurchie-Davidson in 64 bits with
plain torch, without any code of this repository.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

import libint_amd as la
from libint_amd import flop_model

EPS = float(np.finfo(float).eps)
ANGSTROM = 1.0 / 0.529177210903
RECIPES = {
    "plain": [(0, 6), (0, 1), (0, 1), (1, 3), (1, 1), (2, 1)],
    "spd": [(0, 0)] * 4 + [(1, 0)] * 3 + [(2, 0)] * 2,
    "spdf": [(0, 0)] * 4 + [(1, 0)] * 3 + [(2, 0)] * 2 + [(3, 0)],
}
EXPONENTS = {0: (0.1, 5e3), 1: (0.1, 300.0), 2: (0.15, 30.0), 3: (0.25, 8.0)}


def listed():
    return [
        # one quartet per call, as a program that loops over Engine::compute
        dict(name="quartet_call", kind="call", l1=2, l2=1, l3=1, l4=0, kmax=3),
        # every unique quartet of a small molecule in a double-zeta-like basis: conventional SCF
        dict(name="eri_plain10", kind="eri", recipe="plain", natoms=10, kmax=6, nq=0, ls="012"),
        # one heavy class of a contracted basis, the repository's headline class
        dict(name="eri_dddd", kind="eri", recipe="spd", natoms=60, kmax=6, nq=100000, ls="2"),
        # every class up to (ff|ff), deep contractions, random shell order: integral-direct correlation
        dict(name="eri_spdf", kind="eri", recipe="spdf", natoms=40, kmax=8, nq=60000, ls="0123"),
        # weak quartets in the mixed FP32/FP64 mode
        dict(name="eri_mixed", kind="mixed", recipe="spd", natoms=60, kmax=6, nq=500000, ls="12"),
        # short-range Coulomb of range-separated hybrids
        dict(name="eri_erfc", kind="erfc", recipe="spd", natoms=30, kmax=6, nq=100000, ls="012"),
        # density fitting: (X|ab)
        dict(name="eri_3centre", kind="3c", recipe="spd", natoms=30, kmax=6, nq=300000, ls="012"),
        # nuclear gradients: 12 derivative sets a quartet
        dict(name="grad_spd", kind="grad", recipe="spd", natoms=20, kmax=4, nq=20000, ls="012"),
        # core Hamiltonian and overlap at the start of an SCF
        dict(name="onebody_spd", kind="onebody", recipe="spd", natoms=20, kmax=6),
        # J/K builds of an SCF iteration: a few atoms, where latency counts
        dict(name="fock_plain3", kind="fock", recipe="plain", natoms=3, kmax=6),
        # ... an ordinary molecule
        dict(name="fock_spd16", kind="fock", recipe="spd", natoms=16, kmax=6),
        # ... and one with f functions
        dict(name="fock_spdf5", kind="fock", recipe="spdf", natoms=5, kmax=8),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["call", "eri", "eri", "eri", "mixed", "erfc", "3c", "grad", "onebody", "fock", "fock"])
    if kind == "call":
        return dict(kind=kind, l1=rng.randint(0, 3), l2=rng.randint(0, 3), l3=rng.randint(0, 3), l4=rng.randint(0, 3),
                    kmax=rng.randint(1, 6))
    if kind == "onebody":
        return dict(kind=kind, recipe="spd", natoms=_log(rng, 2, 20), kmax=rng.randint(1, 6))
    if kind == "fock":
        recipe = rng.choice(["plain", "spd", "spdf"])
        most = {"plain": 16, "spd": 14, "spdf": 5}[recipe]
        return dict(kind=kind, recipe=recipe, natoms=_log(rng, 2, most), kmax=rng.randint(1, 6))
    if kind == "eri":
        ls = rng.choice(["0123", "012", "23", "2", "12", "01", "3"])
        return dict(kind=kind, recipe="spdf" if "3" in ls else "spd", natoms=rng.randint(10, 60), kmax=rng.randint(1, 6),
                    nq=_log(rng, 500, 60000 if "3" not in ls else 30000 if len(ls) > 2 else 4000), ls=ls)
    if kind == "mixed":
        return dict(kind=kind, recipe="spd", natoms=rng.randint(20, 60), kmax=rng.randint(1, 5), nq=_log(rng, 50000, 400000),
                    ls="12")
    return dict(kind=kind, recipe="spd", natoms=rng.randint(10, 40), kmax=rng.randint(1, 4),
                nq=_log(rng, 1000, {"erfc": 80000, "3c": 250000, "grad": 10000}[kind]), ls="012")


# ---------------------------------------------------------------------------
# molecules and quartet lists (host, numpy)
# ---------------------------------------------------------------------------


def _dfact(n):  # n!! for odd n
    return 1.0 if n <= 1 else n * _dfact(n - 2)


def _normalised(l, alpha, c):
    """Coefficients of primitives x^l-normalised, the contraction scaled to unit self-overlap."""
    c = c * np.sqrt(2.0 ** l * (2 * alpha) ** (l + 1.5) / (math.pi ** 1.5 * _dfact(2 * l - 1)))
    s = math.pi ** 1.5 * _dfact(2 * l - 1) / 2.0 ** l * (np.outer(c, c) / np.add.outer(alpha, alpha) ** (l + 1.5)).sum()
    return c / math.sqrt(s)


def _shell(r, l, K, origin):
    """One shell (l, alpha, c, origin) of K primitives, exponents log-uniform in the range of its l."""
    lo, hi = EXPONENTS[l]
    alpha = np.exp(r.uniform(math.log(lo), math.log(hi), K))
    return l, alpha, _normalised(l, alpha, r.uniform(0.1, 1.0, K)), origin


def _molecule(case, seed):
    """(shells, atom coordinates in bohr); shell: (l, alpha, c, origin).  The case gives the arrangement of the
    atoms and the depth of each shell; the seed moves every atom by up to 0.05 A an axis and draws exponents and
    coefficients, so that the shapes of a case are the same for every seed."""
    r = np.random.default_rng(17)
    n, box = case["natoms"], 14.0 * (case["natoms"] / 60.0) ** (1.0 / 3.0)
    pts = []
    while len(pts) < n:
        p = r.uniform(0.0, box, 3)
        if all(np.linalg.norm(p - o) >= 1.0 for o in pts):
            pts.append(p)
    depth = [(a, l, K or int(r.integers(1, case["kmax"] + 1))) for a in range(n) for l, K in RECIPES[case["recipe"]]]
    r = np.random.default_rng([19, seed])
    xyz = (np.array(pts) + r.uniform(-0.05, 0.05, (n, 3))) * ANGSTROM
    return [_shell(r, l, K, xyz[a]) for a, l, K in depth], xyz


def _basis(shells):
    return la.BasisArrays([s[0] for s in shells], [1 if s[0] >= 2 else 0 for s in shells], [len(s[1]) for s in shells],
                          np.concatenate([s[1] for s in shells]), np.concatenate([s[2] for s in shells]),
                          np.array([s[3] for s in shells]))


def _pair_bounds(shells, only=None):
    """A Schwarz-like size of every shell pair (of the shells `only`) from its s-type Gaussian products."""
    only = range(len(shells)) if only is None else only
    K = max(len(shells[i][1]) for i in only)
    alpha, c = np.ones((len(only), K)), np.zeros((len(only), K))
    for x, i in enumerate(only):
        alpha[x, : len(shells[i][1])], c[x, : len(shells[i][1])] = shells[i][1], np.abs(shells[i][2])
    o, l = np.array([shells[i][3] for i in only]), np.array([shells[i][0] for i in only])
    out = np.zeros((len(shells), len(shells)))
    for x, i in enumerate(only):
        a, b = alpha[x][:, None, None], alpha[: x + 1][None]
        g = a + b
        f = c[x][:, None, None] * c[: x + 1] * np.exp(-a * b / g * ((o[x] - o[: x + 1]) ** 2).sum(1)[:, None]) / g ** 1.25
        row = 5.9 * (f * (0.5 / g) ** (0.5 * (l[x] + l[: x + 1]))[:, None]).max((0, 2))
        out[i, np.array(only[: x + 1])] = row
        out[np.array(only[: x + 1]), i] = row
    return out


def _quartets(case):
    """(n, 4) shell indices of a batch: those that are significant with the exponents of seed 0."""
    shells, _ = _molecule(case, 0)
    keep = [i for i, s in enumerate(shells) if str(s[0]) in case["ls"]]
    K = _pair_bounds(shells, keep)
    i, j = (np.array(keep)[x] for x in np.tril_indices(len(keep)))
    ok = K[i, j] > 1e-8
    p = np.stack([i[ok], j[ok]], 1)
    k = K[p[:, 0], p[:, 1]]
    if not case["nq"]:  # every unique one that a Fock build would keep
        a, b = np.tril_indices(len(p))
        a, b = a[k[a] * k[b] > 1e-12], b[k[a] * k[b] > 1e-12]
        return np.concatenate([p[a], p[b]], 1).astype(np.int32)
    r = np.random.default_rng(23)
    if case["kind"] == "3c":  # (X unit|a b); the unit shell is the last of the basis
        x = r.choice(keep, case["nq"])
        ab = p[r.integers(0, len(p), case["nq"])]
        return np.concatenate([x[:, None], np.full((len(x), 1), len(shells)), ab], 1).astype(np.int32)
    if case["kind"] == "mixed":  # (dp|dp), one class as a class-sorted batch has it
        d, p1 = (np.array([x for x in keep if shells[x][0] == m]) for m in (2, 1))
        p = np.stack([x.ravel() for x in np.meshgrid(d, p1, indexing="ij")], 1)
        p = p[K[p[:, 0], p[:, 1]] > 1e-7]
        s = r.integers(0, len(p), (2, case["nq"]))
        return np.concatenate([p[s[0]], p[s[1]]], 1).astype(np.int32)
    got, n = [], 0
    while n < case["nq"]:
        a, b = r.integers(0, len(p), (2, 2 * case["nq"]))
        fine = k[a] * k[b] > 1e-10
        got.append(np.concatenate([p[a[fine]], p[b[fine]]], 1))
        n += len(got[-1])
    q = np.concatenate(got)[: case["nq"]]
    flip = r.integers(0, 2, (3, len(q))).astype(bool)  # callers give shells in any order
    q[flip[0]] = q[flip[0]][:, [1, 0, 2, 3]]
    q[flip[1]] = q[flip[1]][:, [0, 1, 3, 2]]
    q[flip[2]] = q[flip[2]][:, [2, 3, 0, 1]]
    return q.astype(np.int32)


UNIT = (0, np.zeros(1), np.ones(1), np.zeros(3))


def _batch(case, seed):
    shells, _ = _molecule(case, seed)
    q = _quartets(case)
    return (shells + [UNIT] if case["kind"] == "3c" else shells), q


def _call_shells(case, seed):
    r = np.random.default_rng([29, seed])
    return [_shell(r, case["l%d" % k], case["kmax"], r.uniform(-1.0, 1.0, 3)) for k in (1, 2, 3, 4)]


def _density(nbf, seed):
    C = np.random.default_rng([31, seed]).normal(0.0, 0.1, (nbf, max(1, nbf // 5)))
    return C @ C.T


# ---------------------------------------------------------------------------
# the framework's calls
# ---------------------------------------------------------------------------


def prepare(case, seed):
    kind, ctx = case["kind"], la.default_context()
    if kind == "call":
        shells = [la.Shell(l, list(zip(a, c)), o, pure=l >= 2, renorm=False) for l, a, c, o in _call_shells(case, seed)]
        return dict(kind=kind, engine=la.Engine(case["kmax"], 3, ctx=ctx), shells=shells)
    if kind in ("onebody", "fock"):
        shells, xyz = _molecule(case, seed)
        basis = la.Basis(ctx, _basis(shells))
        if kind == "onebody":
            return dict(kind=kind, basis=basis, charges=[(float(1 + a % 9), tuple(x)) for a, x in enumerate(xyz)])
        fock = la.FockBuilder(basis)
        return dict(kind=kind, fock=fock, D=_density(fock.nbf, seed))
    shells, q = _batch(case, seed)
    basis = la.Basis(ctx, _basis(shells))
    if kind == "grad":
        plan = la.Deriv1Plan(basis, q)
        return dict(kind=kind, plan=plan, out=torch.empty((12, plan.size), dtype=torch.float64, device="cuda"))
    plan = la.EriPlan(basis, q, fp32_threshold=1e-6 if kind == "mixed" else 0.0)
    if kind == "erfc":
        plan.set_operator(la.ERFC_COULOMB, 0.4)
    return dict(kind=kind, plan=plan, out=torch.empty(plan.size, dtype=torch.float64, device="cuda"))


def run(state):
    kind = state["kind"]
    if kind == "call":
        return state["engine"].compute(*state["shells"])
    if kind == "onebody":
        return la.one_body(state["basis"], state["charges"])
    if kind == "fock":
        return state["fock"].build(state["D"], 1e-12)
    state["plan"].execute(state["out"].data_ptr())
    return state["out"]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------


def _size(l):
    return 2 * l + 1 if l >= 2 else (l + 1) * (l + 2) // 2


def _canonical(l):
    b, k = sorted(l[:2], reverse=True), sorted(l[2:], reverse=True)
    return tuple(b + k) if sum(b) <= sum(k) else tuple(k + b)


def work(case):
    """Bytes: the outputs, written once (with the density of a J/K build).  FLOPs: the repository's
    Head-Gordon-Pople count per primitive quartet and per quartet.  Both for the molecule of seed 0."""
    kind = case["kind"]
    if kind == "onebody":
        shells, xyz = _molecule(case, 0)
        n = sum(_size(s[0]) for s in shells)
        prim = sum(len(s[1]) for s in shells) ** 2 / 2
        return {"bytes": 24.0 * n * n, "flops": prim * (len(xyz) * 2000.0 + 500.0)}
    if kind == "call":
        shells, q = _call_shells(case, 0), np.array([[0, 1, 2, 3]])
    elif kind == "fock":
        shells, _ = _molecule(case, 0)
        K = _pair_bounds(shells)
        i, j = np.tril_indices(len(shells))
        ok = K[i, j] > 1e-8
        i, j = i[ok], j[ok]
        o = np.argsort(-K[i, j])
        i, j, k = i[o], j[o], K[i[o], j[o]]
        last = np.searchsorted(-k, -1e-11 / k, side="right")  # partners of each pair, itself and smaller ones
        return _fock_work(shells, i, j, last)
    else:
        shells, q = _batch(case, 0)
    l, K = np.array([s[0] for s in shells]), np.array([len(s[1]) for s in shells])
    lq, code = l[q], l[q] @ np.array([1000, 100, 10, 1])
    prim = K[q].prod(1).astype(float)
    flops = out = 0.0
    for c in np.unique(code):
        at = code == c
        ls = tuple(int(x) for x in lq[at][0])
        n, p = int(at.sum()), float(prim[at].sum())
        flops += flop_model.class_flops(*_canonical(ls), n, p)
        out += 8.0 * n * math.prod(_size(x) for x in ls)
    if kind == "grad":  # each set costs about one integral set of the raised quartet
        return {"bytes": 12 * out, "flops": 8 * flops}
    return {"bytes": out, "flops": flops * (2 if kind == "erfc" else 1)}


def _fock_work(shells, i, j, last):
    l, K = np.array([s[0] for s in shells]), np.array([len(s[1]) for s in shells])
    hi, lo = np.maximum(l[i], l[j]), np.minimum(l[i], l[j])
    types = sorted(set(zip(hi.tolist(), lo.tolist())))
    t = np.array([types.index(x) for x in zip(hi.tolist(), lo.tolist())])
    kk = (K[i] * K[j]).astype(float)
    n_of = np.concatenate([np.zeros((1, len(types))), np.cumsum(np.eye(len(types))[t], 0)])
    p_of = np.concatenate([np.zeros((1, len(types))), np.cumsum(np.eye(len(types))[t] * kk[:, None], 0)])
    at = np.arange(len(i))
    last = np.minimum(last, at + 1)
    flops = 0.0
    for a in range(len(types)):
        m = t == a
        for b in range(len(types)):
            n, p = n_of[last[m], b].sum(), (p_of[last[m], b] * kk[m]).sum()
            c = _canonical(types[a] + types[b])
            flops += flop_model.class_flops(*c, n, p) + n * flop_model.fock_digest_flops(*c)
    nbf = sum(_size(x) for x in l)
    return {"bytes": 32.0 * float(nbf) ** 2, "flops": float(flops)}


# ---------------------------------------------------------------------------
# the same in 64 bits: McMurchie-Davidson in plain torch
# ---------------------------------------------------------------------------


def _carts(l):
    return [(x, y, l - x - y) for x in range(l, -1, -1) for y in range(l - x, -1, -1)]


def _harmonics(l):
    """(functions, Cartesian components) of a shell: real solid harmonics m = -l .. l for l >= 2."""
    at = {c: k for k, c in enumerate(_carts(l))}
    if l < 2:
        return torch.eye(len(at), dtype=torch.float64)
    s3, s6, s10, s15 = math.sqrt(3), math.sqrt(6) / 4, math.sqrt(10) / 4, math.sqrt(15)
    rows = {2: [{(1, 1, 0): s3}, {(0, 1, 1): s3}, {(0, 0, 2): 1, (2, 0, 0): -.5, (0, 2, 0): -.5}, {(1, 0, 1): s3},
                {(2, 0, 0): s3 / 2, (0, 2, 0): -s3 / 2}],
            3: [{(2, 1, 0): 3 * s10, (0, 3, 0): -s10}, {(1, 1, 1): s15},
                {(0, 1, 2): 4 * s6, (2, 1, 0): -s6, (0, 3, 0): -s6},
                {(0, 0, 3): 1, (2, 0, 1): -1.5, (0, 2, 1): -1.5},
                {(1, 0, 2): 4 * s6, (3, 0, 0): -s6, (1, 2, 0): -s6},
                {(2, 0, 1): s15 / 2, (0, 2, 1): -s15 / 2}, {(3, 0, 0): s10, (1, 2, 0): -3 * s10}]}[l]
    m = torch.zeros((len(rows), len(at)), dtype=torch.float64)
    for k, row in enumerate(rows):
        for c, v in row.items():
            m[k, at[c]] = v
    return m


def _hermites(L):
    return [(t, u, v) for t in range(L + 1) for u in range(L + 1 - t) for v in range(L + 1 - t - u)]


def _boys(L, T):
    """[F_0(T), .., F_L(T)]: the ascending series and downward recursion, or erf and upward recursion."""
    big = T > 40.0
    t = torch.where(big, torch.ones_like(T), T)
    term = torch.full_like(t, 1.0 / (2 * L + 1))
    s = term.clone()
    for k in range(1, int(float(t.max()) * 2.2) + 50 if t.numel() else 1):
        term = term * (2 * t / (2 * L + 2 * k + 1))
        s += term
    e = torch.exp(-t)
    low = [s * e]
    for m in range(L, 0, -1):
        low.append((2 * t * low[-1] + e) / (2 * m - 1))
    low.reverse()
    t = torch.where(big, T, torch.full_like(T, 50.0))
    e = torch.exp(-t)
    up = [0.5 * torch.sqrt(math.pi / t) * torch.erf(torch.sqrt(t))]
    for m in range(L):
        up.append(((2 * m + 1) * up[-1] - e) / (2 * t))
    return [torch.where(big, b, a) for a, b in zip(low, up)]


def _hermite_integrals(L, alpha, PQ, pre, omega=None, short=False):
    """{(t,u,v): R_tuv} with (-2 alpha)^n F_n(alpha R^2), alpha (n,), PQ (n, 3)."""
    T = alpha * (PQ * PQ).sum(1)
    F = _boys(L, T)
    if omega is not None:
        s = omega * omega / (omega * omega + alpha)
        G = _boys(L, s * T)
        F = [(f if short else 0.0) + (-1.0 if short else 1.0) * g * s ** (m + 0.5) for m, (f, g) in enumerate(zip(F, G))]
    cur = {}
    f = pre.clone()
    base = []
    for n in range(L + 1):
        base.append(F[n] * f)
        f = f * (-2.0 * alpha)
    for n in range(L, -1, -1):  # level n holds every (t,u,v) with t+u+v <= L - n
        new = {(0, 0, 0): base[n]}
        for h in sorted(_hermites(L - n), key=sum):
            if sum(h) == 0:
                continue
            ax = next(a for a in range(3) if h[a])
            one = tuple(h[a] - (a == ax) for a in range(3))
            v = PQ[:, ax] * cur[one]
            if one[ax]:
                v = v + one[ax] * cur[tuple(one[a] - (a == ax) for a in range(3))]
            new[h] = v
        cur = new
    return cur


def _expansion(l1, l2, a, b, A, B, K):
    """1D Hermite coefficients E[axis][i][j] = list over t, of primitive pairs (K on the x axis)."""
    p = a + b
    P = (a[:, None] * A + b[:, None] * B) / p[:, None]
    out = []
    for ax in range(3):
        pa, pb, h = P[:, ax] - A[:, ax], P[:, ax] - B[:, ax], 0.5 / p
        one = K if ax == 0 else torch.ones_like(a)
        E = [[None] * (l2 + 1) for _ in range(l1 + 1)]

        def up(src, x):
            n = len(src)
            return [x * src[t] * (t < n) + (h * src[t - 1] if t else 0.0) + ((t + 1) * src[t + 1] if t + 1 < n else 0.0)
                    if t < n else h * src[t - 1] for t in range(n + 1)]
        for i in range(l1 + 1):
            E[i][0] = [one] if i == 0 else up(E[i - 1][0], pa)
            for j in range(1, l2 + 1):
                E[i][j] = up(E[i][j - 1], pb)
        out.append(E)
    return P, out


class _Pairs:
    """Primitive pairs of a list of shell pairs of one (l1, l2): exponents, centres, first primitive of each."""

    def __init__(self, shells, i, j, dev):
        self.l = (shells[i[0]][0], shells[j[0]][0])
        rows, first, at = [], [0], {}
        uniq, self.of = np.unique(np.stack([i, j], 1), axis=0, return_inverse=True)
        for x, y in uniq:
            _, a, ca, A = shells[x]
            _, b, cb, B = shells[y]
            aa, bb = np.repeat(a, len(b)), np.tile(b, len(a))
            c = np.outer(ca, cb).ravel() * np.exp(-aa * bb / (aa + bb) * ((A - B) ** 2).sum())
            rows.append(np.column_stack([aa, bb, c, np.tile(A, (len(c), 1)), np.tile(B, (len(c), 1))]))
            first.append(first[-1] + len(c))
        t = torch.from_numpy(np.concatenate(rows)).to(dev)
        self.of = self.of.reshape(-1)
        self.a, self.b, self.K, self.A, self.B = t[:, 0], t[:, 1], t[:, 2], t[:, 3:6], t[:, 6:9]
        self.first, self.n = np.array(first[:-1]), np.diff(first)
        self.p = self.a + self.b

    def matrices(self, deriv=False):
        """P and the (functions of both, Hermites) matrix of each primitive pair; with deriv the six matrices of d/dA, d/dB."""
        (l1, l2), d = self.l, int(deriv)
        P, E = _expansion(l1 + d, l2 + d, self.a, self.b, self.A, self.B, self.K)
        H = _hermites(l1 + l2 + d)
        T = torch.kron(_harmonics(l1), _harmonics(l2)).to(self.a.device)
        zero = torch.zeros_like(self.a)

        def axis(ax, i, j, t, side):
            get = lambda x, y: E[ax][x][y][t] if x >= 0 and y >= 0 and t < len(E[ax][x][y]) else zero  # noqa: E731
            if side == 0:
                return get(i, j)
            if side == 1:
                return 2 * self.a * get(i + 1, j) - i * get(i - 1, j)
            return 2 * self.b * get(i, j + 1) - j * get(i, j - 1)
        out = []
        for side, dx in [(0, -1)] if not deriv else [(s, x) for s in (1, 2) for x in range(3)] + [(0, -1)]:
            tab = [[[[axis(ax, i, j, t, side if ax == dx else 0) for t in range(l1 + l2 + d + 1)] for j in range(l2 + 1)]
                    for i in range(l1 + 1)] for ax in range(3)]
            M = torch.stack([torch.stack([tab[0][c[0]][e[0]][t] * tab[1][c[1]][e[1]][u] * tab[2][c[2]][e[2]][v]
                                          for t, u, v in H], 1) for c in _carts(l1) for e in _carts(l2)], 1)
            out.append(torch.matmul(T, M))
        return P, H, out


def _quartet_values(shells, q, dev, omega=None, deriv=False, most=None):
    """Values of the quartets in the library's layout, one tensor (with deriv: (12, n))."""
    l = np.array([s[0] for s in shells])
    size = np.array([_size(x) for x in l])
    n = size[q].prod(1)
    off = np.concatenate([[0], np.cumsum(n)])
    out = torch.zeros((12 if deriv else 1, int(off[-1])), dtype=torch.float64, device=dev)
    code = l[q] @ np.array([64, 16, 4, 1])
    for c in np.unique(code):
        at = np.nonzero(code == c)[0]
        bra, ket = _Pairs(shells, q[at, 0], q[at, 1], dev), _Pairs(shells, q[at, 2], q[at, 3], dev)
        L = sum(bra.l) + sum(ket.l) + int(deriv)
        Pb, Hb, Mb = bra.matrices(deriv)
        Pk, Hk, Mk = ket.matrices(deriv)
        sign = torch.tensor([(-1.0) ** sum(h) for h in Hk], dtype=torch.float64, device=dev)
        Mk = [(m * sign).transpose(1, 2).contiguous() for m in Mk]
        sets = [(Mb[0], Mk[0])] if not deriv else [(m, Mk[6]) for m in Mb[:6]] + [(Mb[6], m) for m in Mk[:6]]
        Hall = sorted(set(_hermites(L)), key=sum)
        place = {h: k for k, h in enumerate(Hall)}
        take = torch.tensor([[place.get(tuple(x + y for x, y in zip(h, g)), len(Hall)) for g in Hk] for h in Hb], device=dev)
        npb, npk = bra.n[bra.of], ket.n[ket.of]
        w = npb * npk
        step = max(1, int(6e8 // (8 * (len(Hb) * len(Hk) + 3 * len(Hall) + 2 * sets[0][0].shape[1] * len(Hk)))))
        lo = 0
        ends = np.cumsum(w)
        while lo < len(at):
            hi = max(lo + 1, int(np.searchsorted(ends, (ends[lo - 1] if lo else 0) + step, side="right")))
            ww = torch.from_numpy(w[lo:hi]).to(dev)
            which = torch.repeat_interleave(torch.arange(hi - lo, device=dev), ww)
            k = torch.arange(int(w[lo:hi].sum()), device=dev) - torch.repeat_interleave(torch.cumsum(ww, 0) - ww, ww)
            nk = torch.from_numpy(npk[lo:hi]).to(dev)[which]
            x = torch.from_numpy(bra.first[bra.of[lo:hi]]).to(dev)[which] + k // nk
            y = torch.from_numpy(ket.first[ket.of[lo:hi]]).to(dev)[which] + k % nk
            p, r = bra.p[x], ket.p[y]
            R = _hermite_integrals(L, p * r / (p + r), Pb[x] - Pk[y], 2 * math.pi ** 2.5 / (p * r * torch.sqrt(p + r)),
                                   omega, omega is not None)
            R = torch.stack([R[h] for h in Hall] + [torch.zeros_like(p)], 1)[:, take.reshape(-1)].reshape(-1, len(Hb), len(Hk))
            dest = torch.from_numpy(off[at[lo:hi]]).to(dev)
            for s, (mb, mk) in enumerate(sets):
                v = torch.bmm(torch.bmm(mb[x], R), mk[y]).reshape(len(p), -1)
                acc = torch.zeros((hi - lo, v.shape[1]), dtype=torch.float64, device=dev)
                acc.index_add_(0, which, v)
                out[s, (dest[:, None] + torch.arange(v.shape[1], device=dev)[None]).reshape(-1)] = acc.reshape(-1)
            lo = hi
    return out if deriv else out[0]


def _one_body(shells, charges, dev):
    l = [s[0] for s in shells]
    bf = np.concatenate([[0], np.cumsum([_size(x) for x in l])])
    S, T, V = (np.zeros((bf[-1], bf[-1])) for _ in range(3))
    q = torch.tensor([c for c, _ in charges], dtype=torch.float64, device=dev)
    C = torch.tensor(np.array([x for _, x in charges]), device=dev)
    i, j = (x.ravel() for x in np.meshgrid(np.arange(len(l)), np.arange(len(l)), indexing="ij"))
    la_, lb_ = np.array(l)[i], np.array(l)[j]
    for x in sorted(set(zip(la_.tolist(), lb_.tolist()))):
        at = np.nonzero((la_ == x[0]) & (lb_ == x[1]))[0]
        pr = _Pairs(shells, i[at], j[at], dev)
        l1, l2 = pr.l
        P, E = _expansion(l1, l2 + 2, pr.a, pr.b, pr.A, pr.B, pr.K)
        norm, b = (math.pi / pr.p) ** 1.5, pr.b
        tr = torch.kron(_harmonics(l1), _harmonics(l2)).to(dev)
        ov = lambda ax, m, n: E[ax][m][n][0] if n >= 0 else torch.zeros_like(b)  # noqa: E731
        ki = lambda ax, m, n: (-2 * b * b * ov(ax, m, n + 2) + b * (2 * n + 1) * ov(ax, m, n)  # noqa: E731
                               - 0.5 * n * (n - 1) * ov(ax, m, n - 2))
        s = torch.stack([norm * ov(0, c[0], e[0]) * ov(1, c[1], e[1]) * ov(2, c[2], e[2])
                         for c in _carts(l1) for e in _carts(l2)], 1)
        t = torch.stack([norm * sum((ki if a == 0 else ov)(0, c[0], e[0]) * (ki if a == 1 else ov)(1, c[1], e[1])
                                    * (ki if a == 2 else ov)(2, c[2], e[2]) for a in range(3))
                         for c in _carts(l1) for e in _carts(l2)], 1)
        _, H, (M,) = pr.matrices()
        v = torch.zeros_like(s)
        v = torch.matmul(v, tr.T)
        for z, c in zip(q, C):
            R = _hermite_integrals(l1 + l2, pr.p, P - c, -z * 2 * math.pi / pr.p)
            v += torch.bmm(M, torch.stack([R[h] for h in H], 1)[:, :, None])[:, :, 0]
        seg = torch.from_numpy(np.repeat(np.arange(len(pr.n)), pr.n)).to(dev)
        for mat, val in ((S, torch.matmul(s, tr.T)), (T, torch.matmul(t, tr.T)), (V, v)):
            acc = torch.zeros((len(pr.n), val.shape[1]), dtype=torch.float64, device=dev).index_add_(0, seg, val)
            acc = acc.reshape(-1, _size(l1), _size(l2)).cpu().numpy()[pr.of]
            for k, a in enumerate(at):
                mat[bf[i[a]]:bf[i[a] + 1], bf[j[a]]:bf[j[a] + 1]] = acc[k]
    return S, T, V


def _fock(shells, D, dev):
    """G = 2J - K, J, K of every quartet, unscreened."""
    l = np.array([s[0] for s in shells])
    bf = np.concatenate([[0], np.cumsum([_size(x) for x in l])])
    i, j = np.tril_indices(len(shells))
    a, b = np.tril_indices(len(i))
    q = np.stack([i[a], j[a], i[b], j[b]], 1)
    J, K = (torch.zeros_like(torch.from_numpy(D)).to(dev).reshape(-1) for _ in range(2))
    N, d = int(bf[-1]), torch.from_numpy(D).to(dev).reshape(-1)
    code = l[q] @ np.array([64, 16, 4, 1])
    for c in np.unique(code):
        for part in np.array_split(np.nonzero(code == c)[0], 1 + int((code == c).sum()) // 400000):
            qq = q[part]
            n = [_size(x) for x in l[qq[0]]]
            v = _quartet_values(shells, qq, dev).reshape(len(qq), *n)
            o = [torch.from_numpy(bf[qq[:, k]]).to(dev)[:, None] + torch.arange(n[k], device=dev)[None] for k in range(4)]
            deg = np.where(qq[:, 0] == qq[:, 1], 1.0, 2.0) * np.where(qq[:, 2] == qq[:, 3], 1.0, 2.0) \
                * np.where((qq[:, 0] == qq[:, 2]) & (qq[:, 1] == qq[:, 3]), 1.0, 2.0)
            v = v * torch.from_numpy(deg).to(dev)[:, None, None, None, None]
            w, x, y, z = (o[k].reshape([len(qq)] + [n[k] if m == k else 1 for m in range(4)]) for k in range(4))
            for M, f, (r, s), (t, u) in ((J, .5, (w, x), (y, z)), (J, .5, (y, z), (w, x)), (K, .25, (w, y), (x, z)),
                                         (K, .25, (x, z), (w, y)), (K, .25, (w, z), (x, y)), (K, .25, (x, y), (w, z))):
                val = f * v * d[(t * N + u)]
                M.index_add_(0, (r * N + s).expand_as(v).reshape(-1), val.reshape(-1))
    J, K = (0.5 * (M.reshape(N, N) + M.reshape(N, N).T) for M in (J, K))
    return (2 * J - K).cpu().numpy(), J.cpu().numpy(), K.cpu().numpy()


@functools.lru_cache(maxsize=1)
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def exact(case, seed):
    kind, dev = case["kind"], _device()
    if kind == "call":
        return _quartet_values(_call_shells(case, seed), np.array([[0, 1, 2, 3]]), dev).cpu().numpy()
    if kind == "onebody":
        shells, xyz = _molecule(case, seed)
        return _one_body(shells, [(float(1 + a % 9), x) for a, x in enumerate(xyz)], dev)
    if kind == "fock":
        if case["natoms"] > {"plain": 10, "spd": 4, "spdf": 3}[case["recipe"]]:
            return None  # minutes
        shells, _ = _molecule(case, seed)
        return _fock(shells, _density(sum(_size(s[0]) for s in shells), seed), dev)
    shells, q = _batch(case, seed)
    return _quartet_values(shells, q, dev, 0.4 if kind == "erfc" else None, kind == "grad")
