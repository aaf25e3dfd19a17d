"""Edge deltas against the host restatement at the sizes where their ordering
changes: one block sorts up to 8,192 directed records, passes of 8 bits over
the whole key more; every change of one row (a hub), repeats in both
directions, and the two smallest graphs.  CSR arrays: exact.
"""
import numpy as np
import pytest

from tests import graphs, workloads

pytestmark = pytest.mark.gpu

# side of the grid, changes, all at one vertex, weights
CASES = [
    (2, 1, False, False),
    (2, 9, False, True),
    (30, 255, True, True),
    (60, 4095, False, True),
    (60, 4096, True, False),
    (60, 4097, False, True),
    (150, 20000, False, False),
    (150, 20001, True, True),
]


@pytest.mark.parametrize("side,count,hub,weighted", CASES)
def test_delta_of_many_sizes_equals_the_host(gp, ctx, side, count, hub, weighted):
    off, nbr = graphs.grid(side, side)
    n = side * side
    rng = np.random.default_rng(count)
    u = np.full(count, n // 2) if hub else rng.integers(0, n, count)
    v = (u + rng.integers(1, n, count)) % n
    half = count // 2  # the second half repeats the first, reversed, with other weights
    u, v = np.concatenate([u[:count - half], v[:half]]), np.concatenate([v[:count - half], u[:half]])
    u, v = u.astype(np.int32), v.astype(np.int32)
    ins = rng.integers(0, 2, count).astype(np.uint8)
    w = rng.integers(1, 30, count).astype(np.uint32) if weighted else None
    want_off, want_nbr, want_ew = workloads.apply_delta(off, nbr, None, u, v, ins, w)
    g = gp.Graph(ctx, off, nbr)
    try:
        m = gp.apply_delta(ctx, g.h, u, v, ins, w)
        got_off, got_nbr, got_ew, _ = gp.download_graph(ctx, g.h)
        assert m == len(want_nbr)
        assert np.array_equal(got_off, want_off) and np.array_equal(got_nbr, want_nbr)
        assert np.array_equal(got_ew, want_ew if want_ew is not None else np.ones(m, np.uint32))
    finally:
        g.close()
