"""GPU checks of static fields of trees with cell pairs, charges, dipoles and quadrupoles together, against the oracle's
tree field of the same tree, damped and undamped; and of a batch whose leaves are of very different size (whole
snapshots in one leaf beside trees of a few sites a leaf). Bar: 1e-11 of the largest component, that of the
other static-field tests (FP64 sums, here of at most 2,000 terms).
"""
import sys

import numpy as np
import pytest

import oracle as O
from cppe_amd import capi, synthetic

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


class Cut:
    """The first n sites of a water box; its quadrupoles have a trace, which the packing keeps."""

    def __init__(self, n, seed):
        w = synthetic.water_box((n + 2) // 3, seed, anisotropic=True)
        off, idx = w.excl_csr()
        ex = [[e for e in idx[off[i]:off[i + 1]] if e < n] for i in range(n)]
        self.n, self.pos, self.pol, self.iso = n, w.pos[:n], w.pol[:n], w.alpha_iso()[:n]
        self.excl = (np.concatenate([[0], np.cumsum([len(e) for e in ex])]).astype(np.int32),
                     np.array([v for e in ex for v in e], dtype=np.int32))
        self.sources = (w.charges[:n], w.dipoles[:n], w.quadrupoles[:n] + 0.05 * np.array([1, 0, 0, 1, 0, 1]))

    def alpha_iso(self):
        return self.iso

    def excl_csr(self):
        return self.excl

    def reference(self, field, damping):
        q, mu, th = self.sources
        half = th.copy()
        half[:, [0, 3, 5]] *= 0.5
        al = self.iso if damping else None
        F = field(0, q, al, self.excl, damping)
        return F, F - field(1, mu, al, self.excl, damping) + field(2, half, al, self.excl, damping)


def close(F, ref):
    return np.abs(F - ref).max() <= 1e-11 * np.abs(ref).max()


@pytest.mark.parametrize("damping", [0.0, 2.1304])
@pytest.mark.parametrize("n,ncrit,order,theta", [(200, 3, 5, 0.5), (700, 9, 3, 0.7), (1500, 5, 5, 0.3),
                                                 (1500, 33, 7, 0.5), (2000, 64, 5, 0.5), (2000, 200, 4, 0.6)])
def test_tree_fields_of_all_multipoles(n, ncrit, order, theta, damping):
    say("static tree", n, ncrit, order, theta, damping)
    w = Cut(n, 9400 + n)
    S = capi.System(w.pos, alpha_iso=w.iso, excl=w.excl, summation="fmm", ncrit=ncrit, order=order, theta=theta,
                    damping=damping)
    pairs = S.tree_stats()["n_m2l"]
    F, Fq = S.multipole_fields(*w.sources), S.multipole_fields(w.sources[0])
    S.close()
    tree = O.Tree(w.pos, ncrit, order, theta)
    assert pairs == tree.n_m2l > 0
    ref_q, ref = w.reference(tree.field, damping)
    assert close(F, ref) and close(Fq, ref_q)


@pytest.mark.parametrize("damping", [0.0, 2.1304])
@pytest.mark.parametrize("ncrit", [2, 7, 64])
def test_batch_with_leaves_of_very_different_size(ncrit, damping):
    say("static batch", ncrit, damping)
    sizes = [1, 1200, 700, 2, 9, 65, 900, 333]
    direct = [True, True, False, True, False, True, False, True]
    snaps = [Cut(n, 9500 + n) for n in sizes]
    S = capi.Batch(snaps, direct, ncrit=ncrit, damping=damping)
    F = S.split(S.multipole_fields(*(np.concatenate([s.sources[m] for s in snaps]) for m in range(3))))
    Fq = S.split(S.multipole_fields(np.concatenate([s.sources[0] for s in snaps])))
    S.close()
    for s, one, f, fq in zip(snaps, direct, F, Fq):
        tree = None if one else O.Tree(s.pos, ncrit, 5, 0.5)
        field = tree.field if tree else lambda m, src, *rest: O.direct_field(m, s.pos, src, *rest)
        ref_q, ref = s.reference(field, damping)
        assert close(f, ref) and close(fq, ref_q), s.n  # (exactly zero where the reference is)
