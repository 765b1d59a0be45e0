"""GPU checks of small solves without Thole damping against the oracle's pair fields: no damping factor at all, and
sites of no isotropic polarizability among damped ones, whose pairs stay undamped. One site per molecule, so that
the undamped operator is definite (checked). Sizes at the edges of the one-launch solve's three shapes (32, 64 and 128
sites) and one site beyond.

Bars as in the damped solves: the same iteration count, residual norms to 1e-6, moments to 1e-9 of the largest.
"""
import sys

import numpy as np
import pytest

import oracle as O
from cppe_amd import capi, synthetic

pytestmark = pytest.mark.gpu


def system(n, kind):
    w = synthetic.water_box(n, 53 + n, anisotropic=True)
    keep = np.arange(0, 3 * n, 3)
    iso = w.alpha_iso()[keep].copy()
    if kind == "some sites":
        iso[::5] = 0.0
    return w.pos.reshape(-1, 3)[keep].copy(), w.pol[keep], iso, 0.0 if kind == "none" else 2.1304


def full(pol):
    return pol[:, [0, 1, 2, 1, 3, 4, 2, 4, 5]].reshape(-1, 3, 3)


def dense(x, pol, iso, damping):
    """The inverse polarizabilities on the diagonal, less the oracle's field of each unit dipole."""
    n = len(pol)
    B = np.zeros((3 * n, 3 * n))
    for c in range(3 * n):
        m = np.zeros((n, 3))
        m[c // 3, c % 3] = 1.0
        B[:, c] = O.direct_field(1, x, m, iso if damping else None, None, damping)
    for i, a in enumerate(np.linalg.inv(full(pol))):
        B[3 * i:3 * i + 3, 3 * i:3 * i + 3] += a
    return B


def cg(B, pol, rhs, thresh, maxiter):
    al = full(pol)
    amul = lambda v: np.einsum("nij,nj->ni", al, v.reshape(-1, 3)).ravel()
    x = amul(rhs)
    r = rhs - B @ x
    z = amul(r)
    p, norms = z.copy(), []
    for _ in range(maxiter):
        Ap, rz = B @ p, r @ z
        a = rz / (p @ Ap)
        x, r = x + a * p, r - a * Ap
        norms.append(np.linalg.norm(r))
        if norms[-1] < thresh:
            break
        z = amul(r)
        p = z + (z @ r) / rz * p
    return x, norms


@pytest.mark.parametrize("kind", ["none", "some sites"])
@pytest.mark.parametrize("n", [1, 2, 7, 31, 32, 33, 64, 65, 127, 128, 129])
def test_undamped_solves_follow_the_oracle(n, kind):
    print("undamped", n, kind, flush=True)
    sys.stdout.flush()
    x, pol, iso, damping = system(n, kind)
    B = dense(x, pol, iso, damping)
    assert np.linalg.eigvalsh(B)[0] > 0
    rhs = np.random.default_rng(n).normal(size=3 * n) * 0.02
    S = capi.System(x.ravel(), pol, iso, None, summation="direct", damping=damping)
    ref, norms = cg(B, pol, rhs, 1e-9, 100)
    mu, it, dn = S.solve(rhs, thresh=1e-9, maxiter=100)
    y = S.apply_b(rhs)
    S.close()
    assert it == len(norms)
    np.testing.assert_allclose(dn[:it], norms, rtol=1e-6, atol=1e-15)
    np.testing.assert_allclose(mu, ref, rtol=0, atol=1e-9 * np.abs(ref).max())
    np.testing.assert_allclose(y, B @ rhs, rtol=0, atol=1e-11 * np.abs(y).max())
