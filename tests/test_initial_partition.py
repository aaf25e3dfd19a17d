"""The recursive bisection's labels on shapes where its subsets can go wrong:
rows without entries, halves that are empty or fall apart, repeated entries and
self loops, parts that are no power of two (one half is a single part earlier
than the other), two parts (no subset is cut out at all).  The digests are of the
labels of the form that kept no adjacency of its own per subset and looked every
neighbour up in the whole graph.
"""
import hashlib

import numpy as np
import pytest

from tests import graphs


def _messy(n):
    """Self loops, repeated entries, large edge weights and empty rows."""
    rng = np.random.default_rng(n)
    u, v = rng.integers(0, n, (2, 2 * n))
    w = rng.integers(1, 2**31, 2 * n)
    src, dst = np.concatenate([u, v]), np.concatenate([v, u])
    order = np.lexsort((dst, src))
    off = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(src, minlength=n), out=off[1:])
    ew = np.concatenate([w, w])[order]
    return off.astype(np.int32), dst[order].astype(np.int32), ew.astype(np.uint32), rng.integers(1, 9, n).astype(np.uint32)


def _one_heavy(n):
    """A path whose first vertex weighs as much as all others."""
    vw = np.ones(n, np.uint32)
    vw[0] = n
    return graphs.grid(1, n) + (None, vw)


GRAPHS = {
    "path": lambda: graphs.grid(1, 700) + (None, None),
    "grid": lambda: graphs.grid(23, 31) + (None, None),
    "empty": lambda: (np.zeros(301, np.int32), np.zeros(0, np.int32), None, None),
    "hub": lambda: graphs.hub_ring(600, 100, 5),
    "random": lambda: graphs.random_graph(500, 900, 7, 20) + (None,),
    "messy": lambda: _messy(400),
    "one_heavy": lambda: _one_heavy(300),
}
DIGESTS = {
    "empty": {2: "95411ed3963ac7c7", 3: "116f93264ba37929", 5: "e0479eebdc52db33", 16: "634428ee1e474ce7", 37: "cb3c81bad65e520d"},
    "grid": {2: "aa8b65724dba1013", 3: "f8a151ef88c7fd66", 5: "97990df2c3dc830b", 16: "b0980b84ad6408b7", 37: "c6961a284181501c"},
    "hub": {2: "034cd7e9f54c9902", 3: "d00df4833da270ef", 5: "b6ca08ec00a93d23", 16: "212af21a1fca308a", 37: "f477139fd7f14c00"},
    "messy": {2: "85979b4ab7990e05", 3: "48f240d2a93961ef", 5: "2d3e0af0f23202c5", 16: "f17cfe610e112d69", 37: "b6d7e4f9e6bfd619"},
    "one_heavy": {2: "655a3ef0465a9f30", 3: "037ade743da1d06b", 5: "7a2bd460f23eef2e", 16: "655a3ef0465a9f30", 37: "cff3f51248dcccd8"},
    "path": {2: "ae7b5216d730eaf1", 3: "8a714a74be26a4b9", 5: "8adc849550cd65ae", 16: "859afdcd8fe6dfe6", 37: "b2bcc5b627c8127c"},
    "random": {2: "79d4397fc5d1c39c", 3: "1f6a53351695932f", 5: "8fbd08afa39da77b", 16: "67bb93aecb0e6d86", 37: "6972463f2620db7f"},
}


@pytest.mark.parametrize("parts", [2, 3, 5, 16, 37])
@pytest.mark.parametrize("name", sorted(GRAPHS))
def test_labels_of_the_bisection_stay(gp, name, parts):
    if gp.initial_partition_backend() != "bisection":
        pytest.skip("built with another initial partitioner")
    off, nbr, ew, vw = GRAPHS[name]()
    imbalance = 20.0 if name == "one_heavy" else 3.0  # a part has to hold the heaviest vertex
    labels = gp.initial_partition_host(off, nbr, ew, vw, parts, imbalance, 4)
    assert hashlib.sha256(labels.astype(np.int32).tobytes()).hexdigest()[:16] == DIGESTS[name][parts]
