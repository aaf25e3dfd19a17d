"""The edge cut's batch arithmetic on the host: which lanes count an entry and
which row each entry belongs to, at either end of the entry range that a graph
may have (2^31 - 1 entries), full and partly filled batches, one row or many,
rows without entries among them.  Whole numbers: exact.
"""
import numpy as np
import pytest

LAST = 2**31 - 1  # entries of the largest graph


@pytest.mark.parametrize("rows", [1, 2, 63, 256])
@pytest.mark.parametrize("count", [1, 63, 64, 65, 200, 255, 256])
@pytest.mark.parametrize("end", [256, 1 << 20, 2**31 - 256, 2**31 - 100, LAST])
def test_batch_counts_its_own_entries_only(gp, rows, count, end):
    rng = np.random.default_rng(rows * 1000 + count)
    first = end - count
    # Row ends over the batch, some equal (rows without entries); the last row
    # holds the last entry.
    ends = np.sort(rng.integers(first, end + 1, rows))
    ends[-1] = end
    labels = np.arange(rows) % 128
    entries = np.arange(first, end)
    row = np.searchsorted(ends, entries, side="right")
    for other in (labels[row], np.full(count, 127), rng.integers(0, 128, count)):
        assert gp.batch_cut(ends, labels, first, other) == int((labels[row] != other).sum())
