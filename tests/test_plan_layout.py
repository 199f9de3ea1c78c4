"""How ERI plans lay their classes out: which quartets run in pieces, on which
kernel and with how much scratch.  The rules (csrc/launch_rules.h) on the CPU,
the values at the sizes where a rule changes its answer on the GPU."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

import libint_amd as la
import oracle
sys.path.insert(0, os.path.join(os.path.dirname(la.__file__), "codegen"))
import gen_rys  # noqa: E402

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "libint_amd", "csrc")


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def shells(rng, c, ks, pure=True):
    out = []
    for l, k in zip(c, ks):
        a = np.exp(rng.uniform(np.log(0.3), np.log(8.0), k))
        out.append(la.Shell(l, list(zip(a, rng.uniform(0.2, 1.0, k))), tuple(rng.uniform(-0.7, 0.7, 3)),
                            pure=pure and l >= 2))
    return out


def values(plan, split):
    plan.set_wave_split(split)
    plan.execute()
    return plan.download()


def agree(x, y):
    """The integral bar: two summation orders of one contraction."""
    d = np.abs(x - y)
    return not ((d > 1e-12) & (d > 1e-10 * np.abs(y))).any()


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("rules") / "rules")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC,
                    os.path.join(ROOT, "tests", "cpp", "launch_rules_test.cpp"), "-o", exe], check=True)

    def run(*args):
        r = subprocess.run([exe, *map(str, args)], capture_output=True, text=True, check=True)
        return [int(x) for x in r.stdout.split()]
    return run


GIB = 1 << 27  # doubles


def free_memory():
    """Free device memory, from the HIP runtime that the library is linked to."""
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert ctypes.CDLL(la.LIBPATH).hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("cands, cut", [
    ([], []),
    ([(100, 1.0)], [1]),
    ([(2 * GIB, 1.0)], [1]),                                      # the whole of it
    ([(2 * GIB + 1, 1.0)], [0]),
    ([(GIB, 1.0), (GIB, 3.0), (GIB, 2.0)], [0, 1, 1]),            # by gain
    ([(GIB, 3.0), (2 * GIB, 2.0), (GIB, 1.0)], [1, 0, 1]),        # the next that still fits
    ([(GIB, 1.0)] * 58, [1, 1] + [0] * 56),                       # every class at its own limit
])
def test_piece_scratch_of_a_plan_is_bounded(rules, cands, cut):
    got = rules("pieces", 0, *[x for c in cands for x in c])
    assert got == cut
    assert sum(d for (d, _), k in zip(cands, got) if k) <= 2 * GIB


@pytest.mark.gpu
def test_classes_beyond_the_piece_scratch_run_unsplit(ctx):
    """Six f classes of one deep quartet among shallow ones whose pieces take
    0.5 to 0.9 GiB each (a row per quartet at least): together more than
    a plan's 2 GiB.  The plan holds less, and the values are the unsplit ones."""
    rng = np.random.default_rng(6)
    classes = [(3, 3, 3, 3), (3, 2, 3, 3), (3, 2, 3, 2), (2, 2, 3, 3), (3, 1, 3, 3), (2, 2, 3, 2)]
    n = [17000, 22000, 30000, 22000, 26000, 40000]
    sh, q = [], []
    for c, m in zip(classes, n):
        o = len(sh)
        sh += shells(rng, c, (5, 5, 5, 5)) + shells(rng, c, (1, 1, 1, 1))
        q += [[o, o + 1, o + 2, o + 3]] + [[o + 4, o + 5, o + 6, o + 7]] * (m - 1)
    q = np.array(q, np.int32)
    b = la.Basis(ctx, la.BasisArrays.from_shells(sh))
    say(f"case: {len(q)} quartets of six f classes")
    ctx.synchronize()
    free = free_memory()
    plan = la.EriPlan(b, q)
    used = free - free_memory()
    say(f"  plan {used / 2**20:.0f} MiB, cut: {[s['cls'] for s in plan.stats() if s['wave']]}")
    assert 0 < sum(s["wave"] for s in plan.stats()) < 6
    assert used < 2.1 * 2**30  # the pieces, and the lists of 157,000 quartets
    plan.execute()
    v, _ = plan.download()
    w, _ = values(plan, False)
    assert agree(v, w)


@pytest.mark.parametrize("stride", [10 * 10 + 1, 74 * 74 + 1])  # (fs|fs), (ff|ff)
@pytest.mark.parametrize("w", [1, 64, 65, 4096, 2500 ** 2, 46000 ** 2])
def test_a_deep_pair_fits_the_schwarz_window(rules, w, stride):
    pieces, cap = rules("schwarz", w, stride)
    assert 1 <= pieces <= max(1, w) and pieces * stride <= cap
    assert pieces == -(-w // 64) or (pieces + 1) * stride > cap


@pytest.mark.gpu
def test_schwarz_of_a_deep_f_pair(ctx):
    """A pair of 30-primitive f shells, 810,000 primitive quartets: more than
    the 6126 pieces that fit the window at 64 each.  Against the (p|p)
    integrals of an ERI batch, at the integral bar on K^2."""
    rng = np.random.default_rng(8)
    sh = shells(rng, (3, 3), (30, 30))
    b = la.Basis(ctx, la.BasisArrays.from_shells(sh))
    say("case: Schwarz factor of an (f|f) pair of 900 primitive pairs")
    K = la.schwarz(b, np.array([[0, 1]], np.int32), 0.0)
    v, _, _ = la.compute_quartets(b, np.array([[0, 1, 0, 1]], np.int32), precision=0.0)
    assert agree(K ** 2, np.array([np.abs(v).max()]))


@pytest.mark.gpu
def test_pieces_of_a_long_list(ctx):
    """100,000 quartets, one of 4096 primitive quartets, laid out right after
    their lists are sent: the pieces name the quartets of the lists."""
    rng = np.random.default_rng(2)
    sh = shells(rng, (2, 1, 2, 0), (8, 8, 8, 8)) + [x for _ in range(40) for x in shells(rng, (2, 1, 2, 0), (1, 1, 1, 1))]
    q = np.stack([4 * rng.integers(1, 41, 100000) + k for k in range(4)], 1).astype(np.int32)
    q[77777] = (0, 1, 2, 3)
    b = la.Basis(ctx, la.BasisArrays.from_shells(sh))
    say("case: pieces in a list of 100,000 (dp|ds) quartets")
    plan = la.EriPlan(b, q)
    assert any(s["wave"] for s in plan.stats())
    plan.execute()
    v, nz = plan.download()
    w, nw = values(plan, False)
    assert agree(v, w) and np.array_equal(nz, nw)


def test_lanes_per_item(rules):
    """Tiers from len, 4 len and 32 len primitive quartets on; units of 64, 16, 4 and 1 items."""
    assert rules("tiers", 8, 256, 255, 32, 31, 8, 7, 1) == [1, 2, 2, 2, 4]
    assert rules("tiers", 16, *[511] * 5, *[16] * 17, *[15] * 65) == [0, 5, 17, 65, 2 + 2 + 2]
    assert rules("tiers", 8, *[1] * 64) == [0, 0, 0, 64, 1]
    assert rules("tiers", 8, 100000) == [1, 0, 0, 0, 1]
    # by the class alone, and where the batch fills the chip anyway
    assert [rules("length", t, 10 ** 9, 65536, 0)[0] for t in (1, 24, 25, 32, 33, 444)] == [8, 8, 8, 8, 16, 16]
    assert [rules("length", t, 2 * 65536 * 100, 65536, 1)[0] for t in (24, 25, 33)] == [8, 100, 100]
    assert rules("length", 81, 2 * 65536 * 15, 65536, 1) == [16]


def route(rules, c, n, nprim, wmax):
    return bool(rules("faster", *(gen_rys.LANE_COST.get(c) or (0,) * 6), n, nprim, wmax)[0])


@pytest.mark.parametrize("c, n, w, lane", [
    # (class, quartets, primitive quartets each, per-lane kernel): on the sides of the crossings that were measured
    ("1010", 1, 1, True), ("1010", 150000, 1296, True), ("0032", 1, 1, True),
    ("1111", 150000, 1, False), ("1111", 300, 256, False), ("1111", 20000, 256, True), ("1111", 150000, 256, True),
    ("0033", 300, 1, False), ("0033", 20000, 1, True), ("0033", 300, 256, False), ("0033", 60000, 16, True),
    ("1033", 150000, 1, True), ("1033", 150000, 16, False), ("3030", 60000, 256, True), ("3030", 3000, 16, False),
    ("2222", 150000, 1, False), ("2222", 150000, 256, False), ("2121", 10 ** 6, 256, False),  # Rys kernel only
])
def test_which_kernel_a_class_runs_on(rules, c, n, w, lane):
    assert route(rules, c, n, n * w, w) == lane


LANE_CLASSES = sorted(gen_rys.LANE_COST)


def lane_case(c, pure, seed):
    """200 quartets of a class in mixed caller orders: primitive quartets on both sides of the tiers (8, 32, 256 and 16,
    64, 512), solid harmonics or Cartesians."""
    l = [int(x) for x in c]
    rng = np.random.default_rng(seed)
    ks = [(1, 1, 1, 1), (7, 1, 1, 1), (2, 2, 2, 1), (3, 1, 5, 1), (4, 2, 2, 1), (31, 1, 1, 1), (4, 2, 4, 1), (9, 1, 7, 1),
          (4, 4, 2, 2), (15, 1, 17, 1), (4, 4, 4, 4), (7, 1, 73, 1), (8, 4, 4, 4)]
    if sum(l) > 6:
        ks = ks[:8]
    sh = [x for k in ks for x in shells(rng, l, k, pure)]
    q = np.array([[4 * (n % len(ks)) + x for x in range(4)] for n in range(200)], np.int32)
    q[1::3] = q[1::3][:, [1, 0, 2, 3]]
    # (pp|ds) and (ds|pp) are classes of their own
    q[2::3] = q[2::3][:, [1, 0, 3, 2] if l[0] + l[1] == l[2] + l[3] else [2, 3, 1, 0]]
    return la.BasisArrays.from_shells(sh), q[rng.permutation(200)]


@pytest.mark.gpu
@pytest.mark.parametrize("c", LANE_CLASSES)
@pytest.mark.parametrize("pure", [True, False])
def test_per_lane_kernels(ctx, rules, c, pure):
    """Every class that has a per-lane kernel, in a batch that runs on it (the 200 quartets repeated until the rule takes
    it there), each operator, against the oracle: the values of every repeat."""
    arrays, q = lane_case(c, pure, 3 + sum(map(int, c)))
    b = la.Basis(ctx, arrays)
    if c in ("1033", "2033"):  # these only in large batches of shallow quartets
        q = q[(q < 4).all(1)]
    w = arrays.nprim[q].prod(1)
    reps = next(r for r in (1, 50, 150, 400, 1000, 3000) if route(rules, c, r * len(q), r * int(w.sum()), int(w.max())))
    say(f"case: per-lane kernel of ({c}), pure {pure}, {len(q)} quartets {reps} times")
    plan = la.EriPlan(b, np.tile(q, (reps, 1)))
    # reported where the kernel is not the one of the split turned off
    assert reps == 1 or [s["wave"] for s in plan.stats()] == [True]
    for oper, omega in ((la.COULOMB, 0.0), (la.ERF_COULOMB, 0.6), (la.ERFC_COULOMB, 0.6), (la.ERFC_COULOMB, 0.0)):
        plan.set_operator(oper, omega)
        plan.execute()
        g, nz = plan.download()
        o, _, onz = oracle.eri_quartets(arrays, q, **(dict(oper=oper, omega=omega) if oper else {}))
        g = g.reshape(reps, -1)
        assert np.array_equal(nz.reshape(reps, -1), np.tile(onz, (reps, 1)))
        assert all(agree(x, o) for x in (g[0], g[reps // 2], g[-1])), (oper, omega)
        if reps > 1:
            assert agree(g, g[0])
    plan._release()


@pytest.mark.gpu
@pytest.mark.parametrize("c", [c for c in LANE_CLASSES if gen_rys.LANE_COST[c][4] <= 1 and gen_rys.LANE_COST[c][5] <= 1])
def test_light_classes_have_the_same_bits_in_every_batch(ctx, c):
    """With the split off: a quartet alone, among others and from the quartet engine."""
    arrays, q = lane_case(c, True, 11)
    b = la.Basis(ctx, arrays)
    say(f"case: bits of ({c}) quartets")
    plan = la.EriPlan(b, np.tile(q, (40, 1)))
    v, _ = values(plan, False)
    v = v.reshape(40, -1)
    assert (v == v[0]).all()
    off = np.append(la.EriPlan(b, q).offsets(), v.shape[1])
    for k in range(0, 200, 9):
        one = la.EriPlan(b, q[k:k + 1])
        assert np.array_equal(values(one, False)[0], v[0][off[k]:off[k + 1]]), k


@pytest.mark.parametrize("count, nprim, wmax, generic", [
    (100, 4096 + 99, 4096, True), (508, 8 * 4096 + 500, 4096, True), (20, 20 * 4096, 4096, False), (100, 1099, 1000, False),
    (1, 1059, 1059, True), (1, 1058, 1058, False), (4096, 4095 + 4096, 4096, True), (4097, 4096 + 4096, 4096, False),
])
def test_deep_quartets_of_the_largest_classes_unsplit(rules, count, nprim, wmax, generic):
    assert bool(rules("unsplit", count, nprim, wmax)[0]) == generic


@pytest.mark.gpu
@pytest.mark.parametrize("c", ["3233", "3333"])
def test_one_deep_quartet_unsplit(ctx, c):
    """A quartet of 1536 primitive quartets among shallow ones, layout off, against the oracle."""
    l = [int(x) for x in c]
    rng = np.random.default_rng(l[1])
    arrays = la.BasisArrays.from_shells(shells(rng, l, (8, 6, 8, 4)) + shells(rng, l, (1, 1, 1, 1)))
    q = np.array([[4, 5, 6, 7]] * 30 + [[0, 1, 2, 3]], np.int32)
    say(f"case: one deep ({c}) quartet")
    v, nz = values(la.EriPlan(la.Basis(ctx, arrays), q), False)
    o, _, onz = oracle.eri_quartets(arrays, q)
    assert agree(v, o) and np.array_equal(nz, onz)


@pytest.mark.gpu
def test_one_body_matrices_asked_for(ctx):
    """Every choice of S, T and V: the matrices of the call that takes all three, bit for bit."""
    rng = np.random.default_rng(4)
    arrays = la.BasisArrays.from_shells([x for l in (0, 1, 2, 3) for x in shells(rng, (l,), (3,))])
    b = la.Basis(ctx, arrays)
    charges = [(3.0, (0.1, 0.2, 0.3)), (1.0, (-0.4, 0.5, 0.0))]
    full = la.one_body(b, charges)
    n = len(full[0])
    q, xyz = np.array([c[0] for c in charges]), np.array([c[1] for c in charges]).reshape(-1)
    say("case: one-body matrices one by one and in pairs")
    for k in range(1, 8):
        out = [np.zeros((n, n)) if k >> m & 1 else None for m in range(3)]
        rc = la.lib().l2g_onebody(b.handle, 2, q.ctypes.data, xyz.ctypes.data,
                                  *[None if o is None else o.ctypes.data for o in out])
        assert rc == 0
        assert all(o is None or np.array_equal(o, f) for o, f in zip(out, full)), k


# primitive quartets of shells of (a, b, c, d) primitives, on both sides of the tiers (32 and 128) and of the largest
# number of slots that share a quartet; many shallow ones keep the mean below 64, where the generic kernel would take
# the heavy classes
TIER_KS = [(31, 1, 1, 1), (4, 2, 4, 1), (11, 1, 3, 1), (127, 1, 1, 1), (8, 2, 8, 1), (43, 1, 3, 1), (17, 1, 13, 1)]


@pytest.mark.gpu
@pytest.mark.parametrize("c", [(2, 1, 2, 1), (2, 2, 2, 2), (3, 2, 3, 2), (2, 2, 3, 3), (1, 1, 2, 1), (3, 3, 3, 3)])
@pytest.mark.parametrize("pure", [True, False])
def test_slots_of_a_block_share_deep_quartets(ctx, c, pure):
    """Rys kernels unsplit, blocks of 7 to 3 slots in one and in four waves: quartets of the deep tiers next to shallow
    ones, each operator, against the oracle; the same bits in another batch."""
    rng = np.random.default_rng(41 + sum(c))
    ks = TIER_KS if sum(c) < 9 else TIER_KS[:4]
    sh = [x for k in ks for x in shells(rng, c, k, pure)] + shells(rng, c, (1, 1, 1, 1), pure)
    arrays = la.BasisArrays.from_shells(sh)
    deep = np.arange(4 * len(ks), dtype=np.int32).reshape(-1, 4)
    one = np.arange(4 * len(ks), len(sh), dtype=np.int32)[None]
    q = np.concatenate([np.tile(one, (20, 1)), deep, deep[::2]])
    assert (arrays.nprim[q].prod(1)).mean() < 64
    b = la.Basis(ctx, arrays)
    Q = gen_rys.plan(*c).q
    say(f"case: tiers of {c}, pure {pure}, {Q} slots a block")
    over = sum(c) >= 11  # (df|ff) and (ff|ff) report the generic kernel's code on their Rys kernels, too
    for oper, omega in ((la.COULOMB, 0.0), (la.ERF_COULOMB, 0.5), (la.ERFC_COULOMB, 0.5)):
        plan = la.EriPlan(b, q)
        plan.set_operator(oper, omega)
        v, nz = values(plan, False)
        assert over or not any(s["generic"] or s["wave"] for s in plan.stats())
        o, _, onz = oracle.eri_quartets(arrays, q, **(dict(oper=oper, omega=omega) if oper else {}))
        assert agree(v, o) and np.array_equal(nz, onz)
        off = np.append(plan.offsets(), v.size)
        for k in range(20, 20 + len(ks)):
            few = la.EriPlan(b, np.concatenate([q[k:k + 1], np.tile(one, (6, 1))]))
            few.set_operator(oper, omega)
            w = values(few, False)[0]
            assert over or not any(s["generic"] for s in few.stats())
            assert np.array_equal(w[:off[k + 1] - off[k]], v[off[k]:off[k + 1]]), (k, oper)
