"""How ERI plans lay their classes out: which quartets run in pieces, on which
kernel and with how much scratch.  The rules (csrc/launch_rules.h) on the CPU,
the values at the sizes where a rule changes its answer on the GPU."""
import os
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
