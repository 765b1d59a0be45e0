"""GPU checks of untuned systems on a device without room for the lists and blocks of their near-field form: the largest
allocation that succeeds is bounded (cppe_hip_test_largest_allocation), between the system's creation, whose arrays
are smaller, and its first apply. Each takes a form that needs less and gives the same result; a form
that was chosen reports the error.

* direct summation of 9,000 sites: 8 MiB, where the reverse blocks of the tiled symmetric form take 30 (15 in FP32)
* a tree of 60,000 sites: 64 MiB, where the reverse slots of the symmetric form take about 120; 32 MB, where the expanded
  lists take 34 and the largest of the vectors that three right-hand sides have in any form 30.2, so that the
  thread-per-target form is left
* the arena: a chunk that cannot grow as it would is made as large as what is asked for
"""
import ctypes
import sys

import numpy as np
import pytest

from cppe_amd import capi, synthetic

pytestmark = pytest.mark.gpu
DAMP = 2.1304


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture
def most():
    f = capi.lib().cppe_hip_test_largest_allocation
    f.argtypes, f.restype = [ctypes.c_longlong], None
    yield f
    f(0)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("summation,waters,limit,left", [("direct", 3000, 1 << 23, False), ("fmm", 20000, 1 << 26, False),
                                                         ("fmm", 20000, 32000000, True)])
def test_forms_that_need_less(summation, waters, limit, left, precision, most):
    say("memory", summation, waters, limit, precision)
    w = synthetic.water_box(waters, 5, anisotropic=True)
    x = np.random.default_rng(1).normal(0.0, 0.05, size=3 * w.n)
    S = capi.System(w.pos, w.pol, w.alpha_iso(), w.excl_csr(), summation=summation, damping=DAMP)
    ref = S.apply_b(x)
    S.close()
    S = capi.System(w.pos, w.pol, w.alpha_iso(), w.excl_csr(), summation=summation, damping=DAMP, precision=precision)
    most(limit)
    out = S.apply_b(x)
    three = S.apply_b_multi(np.array([x, x, -x]))
    most(0)
    bar = (1e-12 if precision == "fp64" else 5e-6) * np.abs(ref).max()
    assert np.abs(out - ref).max() <= bar
    assert np.abs(three - np.array([ref, ref, -ref])).max() <= bar
    assert (S.profile_apply(precision == "mixed", 1)["near_kernel"] < 0) == left  # (forms 0 to 4 do not time it)
    mu, _, _ = S.solve(ref, thresh=1e-8)
    assert np.linalg.norm(ref - S.apply_b(mu)) < 1e-3 * np.linalg.norm(ref)
    S.close()


def test_chosen_form_keeps_the_error(most):
    w = synthetic.water_box(3000, 5, anisotropic=True)
    S = capi.System(w.pos, w.pol, w.alpha_iso(), w.excl_csr(), summation="direct", damping=DAMP)
    S.set_tune(np.array([11, 128, 64, 0, 11, 128, 64, 0], dtype=np.int32))
    most(1 << 20)
    with pytest.raises(capi.CppeHipError, match="memory"):
        S.apply_b(w.pos.ravel())
    most(0)
    assert np.isfinite(S.apply_b(w.pos.ravel())).all()
    S.close()


def test_chunk_of_what_is_asked_for(most):
    w = synthetic.water_box(3000, 5, anisotropic=True)
    ref = None
    for limit in (0, 3 << 20):  # (a chunk beyond 2 MiB is none of the doubled ones)
        most(limit)
        S = capi.System(w.pos, w.pol, w.alpha_iso(), w.excl_csr(), summation="fmm", damping=DAMP)
        F = S.multipole_fields(w.charges, w.dipoles, w.quadrupoles)
        S.close()
        most(0)
        ref = F if ref is None else ref
        np.testing.assert_array_equal(F, ref)
