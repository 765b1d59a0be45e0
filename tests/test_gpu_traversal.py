"""GPU checks of the dual traversal where a list of the first capacity is full and the walk is repeated with a
larger one, in launches of several hundred blocks: the lists are those of the oracle, pair by pair.

Full in turn: the far list and the frontier (theta 0.3, cells of 16), the near list alone (theta 0.3, cells of
8), the frontier alone (60,000 sites at theta 0.4), the near list and the frontier of a tree of tiny leaves.
"""
import sys

import numpy as np
import pytest

import oracle as O
from cppe_amd import capi, synthetic

pytestmark = pytest.mark.gpu


def numbered(geo, meta):
    """Cells of both trees by level and centre: the rank of each."""
    key = np.concatenate([meta[:, 1:2].astype(float), geo[:, :3]], axis=1)
    rank = np.empty(len(key), dtype=np.int64)
    order = np.lexsort(key.T[::-1])
    rank[order] = np.arange(len(key))
    return rank, key[order]


@pytest.mark.parametrize("waters,ncrit,theta,full", [(2500, 16, 0.3, "far"), (1000, 8, 0.3, "near"),
                                                     (20000, 64, 0.4, "frontier"), (200, 2, 0.1, "near")])
def test_lists_after_a_repeated_walk(waters, ncrit, theta, full):
    print("traversal", waters, ncrit, theta, full, flush=True)
    sys.stdout.flush()
    w = synthetic.water_box(waters, 1002, anisotropic=True)
    T = O.Tree(w.pos, ncrit=ncrit, order=2, theta=theta)
    geo, meta, _ = T.cells()
    m2l, p2p = T.lists()
    S = capi.System(w.pos, summation="fmm", ncrit=ncrit, order=2, theta=theta)
    ex, st = S.tree_export(), S.tree_stats()
    S.close()
    if full == "far":  # (what the first walk has room for; of the frontier nothing is reported)
        assert st["n_m2l"] > 512 * st["ncells"] + 4096
    if full == "near":
        assert st["n_p2p"] > 256 * st["nleaves"] + 4096
    rank, cells = numbered(geo, meta)
    drank, dcells = numbered(ex["geo"], ex["meta"])
    np.testing.assert_array_equal(dcells, cells)
    for name, ours, theirs in (("m2l", drank[ex["m2l"]], rank[m2l]), ("p2p", drank[ex["p2p"]], rank[p2p])):
        a, b = (np.sort(v[:, 0] * len(cells) + v[:, 1]) for v in (ours, theirs))
        assert len(a) == len(b), name
        assert np.array_equal(a, b), name
