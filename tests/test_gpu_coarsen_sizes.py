"""Coarsening against the oracle at the sizes where its scans, selections and
ordered admission change form (one tile of 2,048 elements, one block up to
8,192, tiles of 4,096 above; admission chunks of 1,024), with rows without
entries and one target that thousands of vertices ask for.  Exact.
"""
import numpy as np
import pytest

from tests import graphs

pytestmark = pytest.mark.gpu


def _scattered(n):
    """A random graph on the first nine tenths, nothing on the rest."""
    off, nbr, ew = graphs.random_graph(n * 9 // 10, 2 * n, seed=n, max_weight=5)
    return np.concatenate([off, np.full(n - (len(off) - 1), off[-1], np.int32)]), nbr, ew, None


def _hub(n):
    off, nbr, ew, vw = graphs.hub_ring(n, n // 4, seed=n)
    return off, nbr, None, vw


CASES = [("scattered", n, 4) for n in (600, 2048, 2049, 4096, 4097, 8191, 8192, 8193, 12289, 16500)]
CASES += [("hub", n, 2) for n in (1500, 3500, 9500)]


@pytest.mark.parametrize("kind,n,k", CASES)
def test_hierarchy_equals_the_oracle(gp, og, ctx, kind, n, k):
    off, nbr, ew, vw = _scattered(n) if kind == "scattered" else _hub(n)
    oh = og.Hierarchy(off, nbr, ew, vw, og.coarsen_opts(k))
    g = gp.Graph(ctx, off, nbr, ew, vw)
    h = gp.Hierarchy(ctx, g, gp.coarsen_options(k))
    try:
        assert h.levels == oh.levels
        for level in range(h.levels):
            for got, want in zip(h.graph_at(level), oh.graph(level)):
                assert np.array_equal(got, want)
            if level + 1 < h.levels:
                assert np.array_equal(h.map(level), oh.map(level))
    finally:
        h.close()
        g.close()


def test_long_rows_give_their_sort_scratch_back(gp):
    """64 hubs joined to 65,536 vertices in a ring.  The peak of coarsening is
    the contraction's long rows; 59.2 bytes an entry are reserved when the row
    sort's arrays go back to the arena before the sums are laid out, and 62.9
    when they are kept."""
    hubs, n = 64, 65536
    i = np.arange(n)
    ring = np.sort(np.stack([hubs + (i - 1) % n, hubs + (i + 1) % n], 1), 1)
    rows = np.concatenate([np.tile(np.arange(hubs), (n, 1)), ring], 1)
    off = np.concatenate([np.arange(hubs + 1) * n, hubs * n + (i + 1) * (hubs + 2)]).astype(np.int32)
    nbr = np.concatenate([np.tile(hubs + i, hubs), rows.ravel()]).astype(np.int32)
    with gp.Context(0) as own:
        g = gp.Graph(own, off, nbr)
        before = gp.reserved_bytes(own)
        gp.Hierarchy(own, g, gp.coarsen_options(4)).close()
        taken = gp.reserved_bytes(own) - before
        g.close()
    assert taken <= 61 * len(nbr), taken / len(nbr)
