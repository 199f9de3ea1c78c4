"""The Rys-quadrature kernels: the node and weight table against the moments
it has to reproduce (CPU), and the kernels at the sizes where their layout
changes (GPU): batches around the number of quartets a block holds, primitive
counts around the tiers that share a quartet's loop between slots, deep
quartets cut into pieces, and mixed Cartesian and solid-harmonic shells."""
import os
import sys

import numpy as np
import pytest

import libint_amd as la
import oracle
sys.path.insert(0, os.path.join(os.path.dirname(la.__file__), "codegen"))
import gen_rys  # noqa: E402
import rys_table  # noqa: E402


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def nodes(n, T):
    """Nodes and weights as the kernels take them from the table, in FP64."""
    c = rys_table.table(n)
    iv = np.where(T < rys_table.NI, T, 0).astype(int)
    x = 2.0 * (T - iv) - 1.0
    p = c[iv]
    v = p[..., -1]
    for k in range(rys_table.ND - 2, -1, -1):
        v = v * x[:, None, None] + p[..., k]
    big = T >= rys_table.NI
    v[big] = c[rys_table.NI, :, :, 0][None] * np.stack([1 / T[big], 1 / np.sqrt(T[big])], 1)[:, None, :]
    return v[..., 0], v[..., 1]


@pytest.mark.parametrize("n", range(1, rys_table.NRMAX + 1))
def test_table_reproduces_the_moments(n):
    """sum_r w_r u_r^m = F_m(T), m < 2n.  A node has a relative error of about
    2 ulp, so u^m has 2m: with the sum, (4 m + 8) ulp of F_m."""
    rng = np.random.default_rng(n)
    T = np.concatenate([rng.uniform(0, rys_table.NI, 400), rng.uniform(rys_table.NI, 400, 50),
                        [0.0, 1e-14, 1.0, np.nextafter(1.0, 0), 64.0, np.nextafter(128.0, 0), 128.0]])
    u, w = nodes(n, T)
    assert (u > 0).all() and (u < 1).all() and (w > 0).all()
    F = oracle.boys_reference(T, 2 * n - 1)
    F = np.asarray(F).reshape(len(T), 2 * n)
    # the asymptotic rule leaves out the tail beyond t = 1, below exp(-128)
    for m in range(2 * n):
        rel = np.abs((w * u ** m).sum(1) - F[:, m]) / F[:, m]
        assert rel.max() <= (4 * m + 8) * 2.3e-16, (m, rel.max(), T[rel.argmax()])


def test_every_tile_covers_each_component_once():
    for c in gen_rys.ge.canonical_classes(3):
        if not gen_rys.use(*c):
            continue
        p = gen_rys.plan(*c)
        seen = sorted(k for _, i, j in p.tiles for k in {i, j})
        assert seen == list(range(len(p.outer))), c
        for ax, i, j in p.tiles:
            assert all(p.outer[i][a] == p.outer[j][a] for a in range(3) if a != ax), c
        assert sorted(k for x in p.parts for k in x) == list(range(len(p.inner))), c
        assert p.q * p.nl <= p.nt and p.lds_bytes('fock') <= 160 * 1024, c


CLASSES = [(1, 0, 1, 0), (1, 1, 2, 0), (2, 0, 3, 1), (2, 1, 2, 1), (2, 2, 2, 2), (3, 0, 2, 2), (2, 2, 3, 3), (3, 2, 3, 3),
           (3, 3, 3, 3)]


def shells(rng, c, ks, pure):
    out = []
    for l, k in zip(c, ks):
        a = np.exp(rng.uniform(np.log(0.3), np.log(8.0), k))
        out.append(la.Shell(l, list(zip(a, rng.uniform(0.2, 1.0, k))), tuple(rng.uniform(-0.7, 0.7, 3)),
                            pure=pure and l >= 2))
    return out


def check(ctx, arrays, q, **kw):
    b = la.Basis(ctx, arrays)
    plan = la.EriPlan(b, q)
    if kw.get("oper"):
        plan.set_operator(kw["oper"], kw["omega"])
    plan.execute()
    g, nz = plan.download()
    o, off, onz = oracle.eri_quartets(arrays, q, **kw)
    assert np.array_equal(plan.offsets(), off) and np.array_equal(nz, onz)
    d = np.abs(g - o)
    bad = (d > 1e-12) & (d > 1e-10 * np.abs(o))
    assert not bad.any(), d.max()
    return plan


@pytest.mark.gpu
@pytest.mark.parametrize("c", CLASSES)
def test_batches_around_a_block(ctx, c):
    """1, Q - 1, Q, Q + 1 and 2 Q + 1 quartets of K = 2 shells, solid
    harmonics, Cartesians and both in one batch, in mixed caller orders."""
    Q = gen_rys.plan(*c).q
    rng = np.random.default_rng(sum(c))
    sh = [shells(rng, c, (2, 1, 2, 1), pure) for pure in (True, False)]
    arrays = la.BasisArrays.from_shells(sh[0] + sh[1])
    for mix in ((0,), (1,), (0, 1)):
        for n in sorted({1, Q - 1, Q, Q + 1, 2 * Q + 1} - {0}):
            say(f"case: {c} {n} quartets (block of {Q}), shells {mix}")
            q = np.array([[4 * mix[(k * 7 + x) % len(mix)] + x for x in range(4)] for k in range(n)], np.int32)
            q[1::3] = q[1::3][:, [1, 0, 2, 3]]
            q[2::3] = q[2::3][:, [2, 3, 1, 0]]
            check(ctx, arrays, q)


@pytest.mark.gpu
@pytest.mark.parametrize("c", [(1, 0, 2, 1), (2, 1, 2, 1), (2, 2, 2, 2), (3, 2, 3, 2)])
def test_primitive_tiers(ctx, c):
    """Primitive counts on both sides of the tiers (32 and 128), alone and in
    one batch with the attenuated operators; a quartet has the same bits in
    every batch."""
    rng = np.random.default_rng(7 + sum(c))
    ks = [(1, 1, 1, 1), (31, 1, 1, 1), (4, 2, 4, 1), (11, 1, 3, 1), (127, 1, 1, 1), (8, 2, 8, 1), (43, 1, 3, 1),
          (6, 6, 6, 6)]
    if max(c) > 2:
        ks = ks[:3] + ks[-3:-1]
    sh = [x for k in ks for x in shells(rng, c, k, True)]
    arrays = la.BasisArrays.from_shells(sh)
    q = np.arange(len(sh), dtype=np.int32).reshape(-1, 4)
    say(f"case: {c} primitive counts {[int(np.prod(k)) for k in ks]}")
    for oper, omega in ((la.COULOMB, 0.0), (la.ERF_COULOMB, 0.5), (la.ERFC_COULOMB, 0.5)):
        kw = dict(oper=oper, omega=omega) if oper else {}
        plan = check(ctx, arrays, q, **kw)
        plan.set_wave_split(False)  # no pieces: a quartet's values depend on the quartet only
        plan.execute()
        v, _ = plan.download()
        off = np.append(plan.offsets(), v.size)
        for k in range(len(q)):
            one = la.EriPlan(plan.basis, q[k:k + 1])
            one.set_wave_split(False)
            if oper:
                one.set_operator(oper, omega)
            if not any(s["generic"] for s in one.stats() + plan.stats()):
                one.execute()
                assert np.array_equal(one.download()[0], v[off[k]:off[k + 1]]), (k, oper)


@pytest.mark.gpu
def test_pieces_and_erfc_of_deep_quartets(ctx):
    """Quartets of 10^4 primitives cut into pieces, next to shallow ones."""
    rng = np.random.default_rng(3)
    sh = shells(rng, (2, 2, 2, 1), (10, 10, 10, 10), True) + shells(rng, (2, 2, 2, 1), (1, 1, 1, 1), False)
    arrays = la.BasisArrays.from_shells(sh)
    q = np.array([[0, 1, 2, 3], [4, 5, 6, 7], [3, 0, 1, 2], [0, 5, 2, 7], [2, 2, 1, 3], [7, 4, 5, 6]], np.int32)
    say("case: pieces of deep (dp|dd) quartets")
    for oper, omega in ((la.COULOMB, 0.0), (la.ERFC_COULOMB, 0.7)):
        plan = check(ctx, arrays, q, **(dict(oper=oper, omega=omega) if oper else {}))
        assert any(s["wave"] for s in plan.stats())


def fock_check(ctx, sh, seed):
    """J/K of a random symmetric D against the oracle.  At precision 1e-12 each
    screened-out quartet of the at most 1e3 leaves less than 1e-12 per
    element, and the sums of at most 1e4 terms of order one round below it."""
    arrays = la.BasisArrays.from_shells(sh)
    n = int(arrays.sizes().sum())
    D = np.random.default_rng(seed).normal(0.0, 0.3, (n, n))
    D = D + D.T
    G, J, K = la.FockBuilder(la.Basis(ctx, arrays)).build(D, 1e-12)
    Go, Jo, Ko, _ = oracle.fock_2e(arrays, D, 1e-12)
    for x, y in ((G, Go), (J, Jo), (K, Ko)):
        assert np.abs(x - y).max() <= 1e-9


@pytest.mark.gpu
@pytest.mark.parametrize("gauss", [False, True])
@pytest.mark.parametrize("pure", [(1,), (0,), (0, 1)])
def test_fock_digest_shapes(ctx, pure, gauss):
    """Blocks of solid-harmonic quartets (unrolled digest), of Cartesian ones
    and of both (general loops), in both function orders."""
    rng = np.random.default_rng(17)
    sh = []
    for k, l in enumerate((0, 1, 2, 2, 3, 1)):
        sh += shells(rng, (l,), (2 - k % 2,), bool(pure[k % len(pure)]))
    say(f"case: Fock digest, {pure}, Gaussian order {gauss}")
    ctx.set_solid_harmonics_ordering(la.SHG_GAUSSIAN if gauss else la.SHG_STANDARD)
    oracle.set_shg_ordering(gauss)
    try:
        fock_check(ctx, sh, 5)
    finally:
        ctx.set_solid_harmonics_ordering(la.SHG_STANDARD)
        oracle.set_shg_ordering(False)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 2, 9, 10])
def test_fock_quartet_list_sizes(ctx, n):
    """Quartet lists of 1, 6, 1035 and 1540: one enumeration block holds 1024;
    two builds on one builder share its workspaces."""
    rng = np.random.default_rng(n)
    sh = [x for k in range(n) for x in shells(rng, (k % 3,), (1 + k % 2,), True)]
    say(f"case: Fock build of {n} shells")
    fock_check(ctx, sh, n)
    arrays = la.BasisArrays.from_shells(sh)
    fb = la.FockBuilder(la.Basis(ctx, arrays))
    N = int(arrays.sizes().sum())
    one = [fb.build(s * np.eye(N), 1e-12) for s in (1.0, 1e-3, 1.0)]
    for x, y in zip(one[0], one[2]):
        assert np.abs(x - y).max() <= 1e-9


@pytest.mark.gpu
@pytest.mark.parametrize("c", [(1, 0, 2, 1), (2, 1, 2, 1)])
def test_fp32_lane_tiers(ctx, c):
    """The per-lane FP32 kernels share a quartet between 1, 4, 16 or 64 lanes
    from 16, 64 and 512 primitive quartets on.  n additions in FP32 round by
    at most n eps of the pre-HRR size S_ab S_cd; a lost or doubled primitive
    of 513 would be off by 2e-3 of the value."""
    rng = np.random.default_rng(5 + sum(c))
    ks = [(5, 3, 1, 1), (16, 1, 1, 1), (17, 1, 1, 1), (9, 7, 1, 1), (8, 1, 8, 1), (13, 1, 5, 1), (73, 1, 7, 1),
          (16, 2, 16, 1), (27, 1, 19, 1)]
    sh = [x for k in ks for x in shells(rng, c, k, True)]
    b = la.Basis(ctx, la.BasisArrays.from_shells(sh))
    q = np.arange(len(sh), dtype=np.int32).reshape(-1, 4)
    say(f"case: FP32 {c} primitive counts {[int(np.prod(k)) for k in ks]}")
    ctx.set_fp32_policy(la.FP32_ALWAYS)
    try:
        m = la.EriPlan(b, q, fp32_threshold=1e6)
        assert all(s["fp32"] for s in m.stats())
    finally:
        ctx.set_fp32_policy(la.FP32_MEASURED)
    m.execute()
    g, _ = m.download()
    o, off, _ = oracle.eri_quartets(b.arrays, q)
    _, S = la.precision_bounds(b, np.concatenate([q[:, :2], q[:, 2:]]))
    ends = np.append(off[1:], o.size)
    for k in range(len(q)):
        bar = (np.prod(ks[k]) + 16) * 1.2e-7 * S[k] * S[k + len(q)]
        assert np.abs(g[off[k]:ends[k]] - o[off[k]:ends[k]]).max() <= bar, ks[k]


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 7, 8, 9, 16, 17])
def test_one_body_items_around_a_wave(ctx, n):
    """8 primitive pairs of two shells and n charges: 8 n items for 64 lanes."""
    from oracle import onebody
    rng = np.random.default_rng(n)
    sh = shells(rng, (2,), (2,), False) + shells(rng, (1,), (4,), False)
    charges = [(float(z), rng.normal(0, 1.2, 3)) for z in rng.uniform(1, 8, n)]
    say(f"case: one-body integrals, {n} charges")
    got = la.one_body(la.Basis(ctx, la.BasisArrays.from_shells(sh)), charges)
    ref = onebody.one_body([(s.l, s.alpha, s.coeff, s.O) for s in sh], charges)
    for g, o in zip(got, ref):
        d = np.abs(g - o)
        assert not ((d > 1e-12) & (d > 1e-10 * np.abs(o))).any()
