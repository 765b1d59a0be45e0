"""GPU checks of the FP32 arithmetic that untuned mixed-precision systems work in: the error of the field of an apply
against the FP64 one, over sizes, both summations, with and without damping.

It is no larger than that of the thread-per-target form (variant 0), whose place the default forms take: that form
rounds each displacement once, takes the damping of every pair below its cutoff and passes over excluded pairs. Both
errors are roundings that depend on the positions, so their 2-norms are compared as means over boxes; the bar
leaves a tenth for that. Right-hand sides that share an apply and single ones alike.
"""
import sys

import numpy as np
import pytest

from cppe_amd import capi, synthetic

pytestmark = pytest.mark.gpu
GENERAL = np.array([0, 256, 64, 0, 0, 256, 64, 0], dtype=np.int32)


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def errors(waters, seed, summation, damping):
    w = synthetic.water_box(waters, seed, anisotropic=True)
    x = np.random.default_rng(seed).normal(0.0, 0.05, size=3 * w.n)
    kw = dict(summation=summation, damping=damping)
    S = capi.System(w.pos, w.pol, w.alpha_iso(), w.excl_csr(), **kw)
    ref = S.apply_b(x)
    field = ref - S.apply_alpha_inv(x)
    S.close()
    S = capi.System(w.pos, w.pol, w.alpha_iso(), w.excl_csr(), precision="mixed", **kw)
    one = S.apply_b(x)
    three = S.apply_b_multi(np.array([x, 0.5 * x[::-1], x]))[2]
    S.set_tune(GENERAL)
    former = S.apply_b(x)
    S.close()
    return [np.linalg.norm(v - ref) / np.linalg.norm(field) for v in (one, three, former)]


@pytest.mark.parametrize("damping", [2.1304, 0.0])
@pytest.mark.parametrize("summation,waters,boxes", [("direct", 2, 24), ("direct", 6, 16), ("direct", 43, 8),
                                                    ("direct", 100, 8), ("direct", 700, 4), ("direct", 3000, 2),
                                                    ("fmm", 150, 8), ("fmm", 1000, 4), ("fmm", 8000, 2)])
def test_error_of_untuned_applies(summation, waters, boxes, damping):
    e = np.array([errors(waters, 100 * waters + k, summation, damping) for k in range(boxes)]).mean(axis=0)
    say("%s %d waters, damping %g: error of the field %.3g, of three %.3g, thread per target %.3g"
        % (summation, waters, damping, *e))
    assert e[0] < 1.1 * e[2]
    assert e[1] < 1.1 * e[2]
