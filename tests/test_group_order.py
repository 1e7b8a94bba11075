"""The order in which the column kernels give work-groups to the XCDs.  No GPU needed."""
import ctypes

import pytest

from openifs_amd import build as B


@pytest.mark.parametrize("n", [1, 5, 7, 8, 9, 15, 16, 257, 513, 1024, 2047])
def test_order(n):
    """Every group once; an XCD's groups are neighbours, in order; and the last group, which may be padding, is the last of
    the XCD that has most: 131,072 columns in blocks of 100 are 512 groups of 256 and one without a column, and no XCD
    may have 65 full ones."""
    lib = ctypes.CDLL(B.DEVICE_CHECK)
    order = [lib.group_order(i, n) for i in range(n)]
    assert sorted(order) == list(range(n))
    mine = [order[x::8] for x in range(min(8, n))]
    for m in mine:
        assert m == list(range(m[0], m[0] + len(m)))
    most = max(len(m) for m in mine)
    assert n - 1 in [m[-1] for m in mine if len(m) == most]
