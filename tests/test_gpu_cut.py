"""gp_edge_cut and gp_edge_cut_noalloc on shapes where the even split of rows
and entries over the waves can go wrong.  A wave's share is at most 256 steps
(a row is one, an entry is one) until a graph has more than 512 x 4,096 of
them, and grows from there; it walks its entries in windows of 256 rows and
batches of 256 entries.  So: rows without entries (a few, a share's worth, whole
windows inside a share), one row over many shares, row counts around a window,
sizes just below and above 512 x 4,096 steps in byte and int32 labels, weights
whose sum passes 2^32, 2 and 128 parts.  Whole numbers: exact.
"""
import ctypes

import numpy as np
import pytest

from tests import graphs

pytestmark = pytest.mark.gpu


class DeviceLabels:
    """Labels in device memory, through the HIP runtime that the library is
    linked with."""

    def __init__(self, gp, labels):
        self.hip, self.size = gp.lib(), labels.nbytes
        self.ptr = ctypes.c_void_p()
        assert self.hip.hipMalloc(ctypes.byref(self.ptr), ctypes.c_size_t(self.size)) == 0
        self.set(labels)

    def set(self, labels):
        host_to_device = 1
        assert self.hip.hipMemcpy(self.ptr, labels.ctypes.data_as(ctypes.c_void_p), ctypes.c_size_t(self.size),
                                  ctypes.c_int(host_to_device)) == 0

    def close(self):
        assert self.hip.hipFree(self.ptr) == 0


def _star(n, isolated_before, isolated_after):
    """A star over n vertices among rows without entries."""
    edges = [(isolated_before, isolated_before + i) for i in range(1, n)]
    off, nbr, _ = graphs.csr_from_edges(isolated_before + n + isolated_after, edges)
    return off, nbr, None, None


def _heavy(n, m):
    off, nbr, ew, vw = graphs.heavy_weights(n, m, 3)
    return off, nbr, ew, vw


def _scattered_edges(n, gap):
    """Three edges, to the next vertex and two across the gap, after every
    `gap` rows without entries."""
    at = np.arange(gap, n - gap, gap, dtype=np.int64)
    u = np.concatenate([at, at, at[:-1] + 1])
    v = np.concatenate([at + 1, at + 2, at[1:]])
    src, dst = np.concatenate([u, v]), np.concatenate([v, u])
    order = np.lexsort((dst, src))
    off = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(src, minlength=n), out=off[1:])
    return off.astype(np.int32), dst[order].astype(np.int32), None, None


CASES = {
    "one_edge": lambda gp: _star(2, 0, 0),
    "edge_after_70_empty_rows": lambda gp: _star(2, 70, 0),
    "edge_before_200_empty_rows": lambda gp: _star(2, 0, 200),
    "star_40000_among_empty_rows": lambda gp: _star(40000, 130, 65),
    "path_33": lambda gp: graphs.grid(1, 33) + (None, None),
    "path_255": lambda gp: graphs.grid(1, 255) + (None, None),
    "path_256": lambda gp: graphs.grid(1, 256) + (None, None),
    "path_257": lambda gp: graphs.grid(1, 257) + (None, None),
    # Shares of 613 steps, windows without an entry before the first edge in
    # one; shares of 864, a window without an entry between two of their edges.
    "edges_every_1500_of_5000000_rows": lambda gp: _scattered_edges(5000000, 1500),
    "edges_every_600_of_7000000_rows": lambda gp: _scattered_edges(7000000, 600),
    # 2,093,690 and 2,100,166 steps: 512 blocks with shares of 256 and 257.
    "grid_647x648": lambda gp: gp.generate_grid(647, 648) + (None, None),
    "grid_648x649": lambda gp: gp.generate_grid(648, 649) + (None, None),
    "grid_64x63": lambda gp: gp.generate_grid(64, 63) + (None, None),
    "grid_129x127": lambda gp: gp.generate_grid(129, 127) + (None, None),
    "grid_520x511": lambda gp: gp.generate_grid(520, 511) + (None, None),  # labels narrowed to bytes
    "rmat13": lambda gp: gp.generate_rmat(13, 9, seed=2) + (None, None),
    "rmat17": lambda gp: gp.generate_rmat(17, 16, seed=5) + (None, None),
    "knn": lambda gp: gp.generate_knn3d(5003, 10, seed=2),
    "heavy_weights": lambda gp: _heavy(300, 4000),
}


@pytest.mark.parametrize("parts", [2, 7, 128])
@pytest.mark.parametrize("name", sorted(CASES))
def test_cut_and_loads_equal_a_recount(gp, ctx, name, parts):
    off, nbr, ew, vw = CASES[name](gp)
    n = len(off) - 1
    rng = np.random.default_rng(n + parts)
    labels = rng.integers(0, parts, n, dtype=np.int32)
    labels[: n // 2] = 0  # a stretch of equal labels
    rows = np.repeat(np.arange(n), np.diff(off))
    weight = np.ones(len(nbr), np.int64) if ew is None else ew.astype(np.int64)
    mass = np.ones(n, np.int64) if vw is None else vw.astype(np.int64)
    want_cut = int(weight[labels[rows] != labels[nbr]].sum()) // 2
    want_loads = np.zeros(parts, np.int64)
    np.add.at(want_loads, labels, mass)
    dev = DeviceLabels(gp, labels)
    g = gp.Graph(ctx, off, nbr, ew, vw)
    try:
        for evaluate in (gp.edge_cut, gp.edge_cut_noalloc, gp.edge_cut):
            cut, loads = evaluate(ctx, g.h, dev.ptr.value, parts)
            assert cut == want_cut
            assert np.array_equal(loads.astype(np.int64), want_loads)
        labels[n - 1] = parts  # one label out of range
        dev.set(labels)
        with pytest.raises(RuntimeError, match="labels outside"):
            gp.edge_cut(ctx, g.h, dev.ptr.value, parts)
    finally:
        g.close()
        dev.close()
