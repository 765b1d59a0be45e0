"""GPU checks of trees whose near lists are not symmetric (theta = 1, where cells of the lattice touch the
acceptance bound and a pair may be far from one side only).

* an untuned FP64 tree of a size that would take the symmetric near field applies and solves as the oracle's tree
* the symmetric form, asked for by name, refuses such a tree whichever side of the pair is missing (one
  one-sided pair in a box and in its mirror images), and agrees with the oracle where the lists are symmetric
* tuning passes over that form
Bars: 1e-11 for an apply and 1e-9 for moments, as for the other trees.
"""
import sys

import numpy as np
import pytest

import oracle as O
from cppe_amd import capi, synthetic

pytestmark = pytest.mark.gpu
DAMP = 2.1304


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


def one_sided(pos, ncrit, theta):
    _, p2p = O.Tree(pos, ncrit=ncrit, order=2, theta=theta).lists()
    pairs = set(map(tuple, p2p))
    return sum((b, a) not in pairs for a, b in pairs)


def test_untuned_tree_of_a_large_system():
    w = synthetic.water_box(20000, 1002, anisotropic=True)
    say("one-sided lists, sites", w.n)
    assert one_sided(w.pos, 64, 1.0) > 0
    S = capi.System(w.pos, w.pol, w.alpha_iso(), w.excl_csr(), summation="fmm", theta=1.0, damping=DAMP)
    B = O.BSystem(w.pos, w.pol, w.excl_csr(), damping=DAMP, scheme="fmm", theta=1.0)
    x = np.random.default_rng(4).normal(0.0, 0.1, size=3 * w.n)
    assert rel(S.apply_b(x), B.apply(x)) < 1e-11
    rhs = np.random.default_rng(5).normal(0.0, 0.02, size=3 * w.n)
    mu, _, _ = S.solve(rhs, thresh=1e-8)
    assert np.linalg.norm(rhs - B.apply(mu)) < 2e-8
    S.close()


@pytest.mark.parametrize("flip", range(8))
def test_symmetric_form_needs_both_sides(flip):
    w = synthetic.water_box(1000, 5, anisotropic=True)
    pos = w.pos.reshape(-1, 3) * [1 - 2 * (flip >> c & 1) for c in range(3)]
    count = one_sided(pos, 8, 1.0)
    say("mirror image", flip, "one-sided pairs", count)
    if flip == 0:
        assert count > 0
    excl = w.excl_csr()
    x = np.random.default_rng(6).normal(0.0, 0.1, size=3 * w.n)
    ref = O.BSystem(pos, w.pol, excl, damping=DAMP, scheme="fmm", ncrit=8, theta=1.0).apply(x)
    for prec, bar in (("fp64", 1e-11), ("mixed", 1e-5)):
        S = capi.System(pos, w.pol, w.alpha_iso(), excl, summation="fmm", ncrit=8, theta=1.0, damping=DAMP,
                        precision=prec)
        assert rel(S.apply_b(x), ref) < bar
        for v in (9, 11):
            S.set_tune(np.array([v, 64, 64, 0, v, 64, 64, 0], dtype=np.int32))
            if count:
                with pytest.raises(capi.CppeHipError):
                    S.apply_b(x)
            else:
                assert rel(S.apply_b(x), ref) < bar
        if count:
            S.autotune(reps=1)
            assert rel(S.apply_b(x), ref) < bar
        S.close()
