"""Capacity repair from lopsided starts against the oracle, at the sizes where
its forms change: one block selects the donors up to 8,192 vertices and tiles
of 4,096 above; one launch admits up to 4,096 eligible donors, up to 1,024 of
them one to a thread, and groups of launches more; destinations come from
prefix sums when a donor is no heavier than the smallest room and from a walk
over the parts otherwise.  Labels, cut and statistics: exact.
"""
import numpy as np
import pytest

from tests import graphs

pytestmark = pytest.mark.gpu


def _path(n, heavy):
    """A path with a chord every 7 vertices; heavy: vertex weights 1..9."""
    edges = [(v, v + 1) for v in range(n - 1)] + [(v, v + 7) for v in range(0, n - 7, 7)]
    off, nbr, _ = graphs.csr_from_edges(n, sorted(set(edges)))
    vw = (np.arange(n, dtype=np.uint32) * 2654435761 >> 7) % 9 + 1 if heavy else None
    return off, nbr, None if vw is None else vw.astype(np.uint32)


# vertices, parts, share of the vertices that start in part 0, weighted
CASES = [
    (60, 2, 0.9, False),
    (1023, 3, 0.7, True),
    (4096, 16, 0.2, False),
    (8191, 128, 0.05, True),
    (8192, 128, 0.3, False),
    (8193, 128, 0.3, True),
    (12288, 5, 0.21, False),
    (12289, 5, 0.5, True),
    (40001, 64, 0.05, True),
    (40001, 64, 0.5, False),
]


@pytest.mark.parametrize("n,k,share,weighted", CASES)
def test_repair_of_a_lopsided_start_equals_the_oracle(gp, og, ctx, n, k, share, weighted):
    off, nbr, vw = _path(n, weighted)
    rng = np.random.default_rng(n + k)
    init = (np.arange(n, dtype=np.int64) * k // n).astype(np.int32)
    init[rng.random(n) < share] = 0
    want, ost = og.refine_graph(off, nbr, None, vw, init, og.refine_opts(k))
    assert ost["repair_moves"] > 0
    g = gp.Graph(ctx, off, nbr, None, vw)
    try:
        got, st = g.refine(init, gp.refine_options(k))
    finally:
        g.close()
    for key in ("initial_repair_failed", "rounds", "initial_cut", "final_cut", "lp_moves", "repair_moves",
                "group_moves", "repair_iterations"):
        assert st[key] == ost[key], key
    assert np.array_equal(got, want)


def test_repair_workspace_does_not_grow_with_the_vertices(gp):
    """A repair of some thousand donors keeps two arrays by vertex: the donor
    list (4 bytes) and its flags (1 byte).  Records, tried parts and connection
    rows go by the donors."""
    n, k, over = 1 << 20, 2, 1000
    off, nbr, _ = _path(n, False)
    init = np.zeros(n, np.int32)
    init[int(1.03 * n / k) + over:] = 1
    with gp.Context(0) as own:
        g = gp.Graph(own, off, nbr, None, None)
        try:
            _, st = g.refine(init, gp.refine_options(k))
            taken = gp.reserved_bytes(own)
        finally:
            g.close()
    assert st["repair_moves"] >= over
    # By vertex: offsets, weights and labels of the caller 12, labels as bytes
    # and their checkpoint 2, state 4, gains 8, five lists and the buckets 24,
    # the repair's two 5: 55.  An array is rounded up by an eighth at most; the
    # connection rows of 4,096 donors and the rest are far below 4 MiB.
    assert taken <= 9 / 8 * (55 * n + 4 * len(nbr)) + (4 << 20), (taken, n, len(nbr))
