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
