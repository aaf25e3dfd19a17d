"""Exchange against the oracle at the list lengths where the ordering of its
moves changes: runs of 256 moves of a part, merged with the keys of eight runs
(2,048 moves) at a time.  A part of a pair has at most 2,048 moves in the
archive and 4,608 in the pool (k <= 32).  Labels, cut and statistics: exact.
"""
import numpy as np
import pytest

from tests import graphs

pytestmark = pytest.mark.gpu

# vertices, edges, largest edge weight, parts, LP rounds, least and most moves
# of one part that the pool has to hold for the case to be what it is here for
CASES = [
    (2000, 6000, 1, 3, 32, 1, 256),
    (3000, 9000, 1, 2, 32, 100, 256),
    (1000, 3000, 1, 3, 1, 257, 2048),
    (6000, 18000, 1, 2, 1, 1500, 2048),
    (2000, 40000, 20, 2, 1, 2049, 4608),
]


@pytest.mark.parametrize("n,m,heaviest,k,rounds,least,most", CASES)
def test_exchange_equals_the_oracle(gp, og, ctx, n, m, heaviest, k, rounds, least, most):
    off, nbr, ew = graphs.random_graph(n, m, seed=n + m, max_weight=heaviest)
    ew = ew if heaviest > 1 else None
    # Unordered starts leave many improving groups after few rounds.
    start = np.arange(n) if rounds > 1 else np.random.default_rng(1).permutation(n)
    init = (start * k // n).astype(np.int32)
    og.most_moves(reset=True)
    want, ost = og.refine_graph(off, nbr, ew, None, init, og.refine_opts(k, max_rounds=rounds))
    assert least <= og.most_moves()[1] <= most
    assert ost["group_moves"] > 0
    g = gp.Graph(ctx, off, nbr, ew, None)
    try:
        got, st = g.refine(init, gp.refine_options(k, max_rounds=rounds))
    finally:
        g.close()
    for key in ("rounds", "initial_cut", "final_cut", "lp_moves", "repair_moves", "group_moves"):
        assert st[key] == ost[key], key
    assert np.array_equal(got, want)
