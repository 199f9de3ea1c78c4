"""Exponents that make no Gaussian are refused before anything is launched: a
primitive pair with a negative sum would give the Boys and node tables a
negative argument."""
import numpy as np
import pytest

import libint_amd as la
import oracle

pytestmark = pytest.mark.gpu


def arrays(alphas):
    rng = np.random.default_rng(1)
    l = np.arange(len(alphas)) % 2
    return la.BasisArrays(l, [0] * len(alphas), [1] * len(alphas), np.array(alphas), np.ones(len(alphas)),
                          rng.uniform(-0.5, 0.5, (len(alphas), 3)))


def test_negative_sum_of_exponents_is_an_error(ctx):
    print("case: negative sums of exponents", flush=True)
    B = arrays([-0.2, 0.1, 1.0, 0.7])
    b = la.Basis(ctx, B)
    q = np.array([[2, 3, 0, 1]], np.int32)
    with pytest.raises(la.L2gError, match="exponents"):
        la.EriPlan(b, q)
    with pytest.raises(la.L2gError, match="exponents"):
        la.schwarz(b, np.array([[0, 1]], np.int32))
    with pytest.raises(la.L2gError, match="exponents"):
        la.FockBuilder(b)
    with pytest.raises(la.L2gError, match="exponent"):
        la.one_body(b, [(1.0, (0.0, 0.0, 0.1))])
    sh = [la.Shell(int(l), [(a, 1.0)], tuple(o), renorm=False) for l, a, o in zip(B.l, B.alpha, B.origin.reshape(-1, 3))]
    with pytest.raises(la.L2gError, match="exponents"):
        la.Engine(1, 1, ctx=ctx).compute(sh[2], sh[3], sh[0], sh[1])


def test_negative_exponent_with_positive_sums(ctx):
    """As before: every primitive pair of this quartet is a Gaussian."""
    print("case: a negative exponent with positive sums", flush=True)
    B = arrays([-0.2, 0.9, 1.0, 0.7])
    q = np.array([[0, 1, 2, 3], [3, 2, 1, 0]], np.int32)
    g, off, nz = la.compute_quartets(la.Basis(ctx, B), q)
    o, _, onz = oracle.eri_quartets(B, q)
    d = np.abs(g - o)
    assert not ((d > 1e-12) & (d > 1e-10 * np.abs(o))).any() and np.array_equal(nz, onz)
