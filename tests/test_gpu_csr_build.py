"""COO -> CSR around the edges of its one-pass kernel: blocks of 4,096 keys, the
256 blocks that one step of the chain takes, runs of empty rows before, between
and after the edges, duplicates that meet at block ends, and nothing kept."""
import numpy as np
import pytest

from back40computing_amd import B40CError, bfs

pytestmark = pytest.mark.gpu

B = 4096


def expected(n, rows, cols, drop, sym):
    r, c = rows.astype(np.int64), cols.astype(np.int64)
    if sym:
        r, c = np.concatenate([r, c]), np.concatenate([c, r])
    if drop:
        keep = r != c
        r, c = r[keep], c[keep]
    key = np.unique(r * n + c)
    return np.searchsorted(key, np.arange(n + 1, dtype=np.int64) * n).astype(np.int32), (key % n).astype(np.int32)


def edges(pattern, n, m, rng):
    if pattern == "dense":
        return rng.integers(0, n, m), rng.integers(0, n, m)
    if pattern == "gaps":  # a few rows in the middle: long empty runs on both sides and between
        return rng.choice(np.array([n // 3, n // 3 + 1, n // 2, n // 2 + 17]) % n, m), rng.integers(0, n, m)
    if pattern == "ends":  # only the first and the last row
        return rng.integers(0, 2, m) * (n - 1), rng.integers(0, n, m)
    if pattern == "same":
        return np.full(m, n // 2), np.full(m, n - 1)
    return (np.arange(m) % n,) * 2  # loops


@pytest.mark.parametrize("m", [0, 1, 63, 65, B - 1, B, B + 1, 256 * B + 1])
@pytest.mark.parametrize("n", [1, 2, 1000, 70001])
@pytest.mark.parametrize("pattern", ["dense", "gaps", "ends", "same", "loops"])
def test_coo_blocks(m, n, pattern):
    rng = np.random.default_rng(m + n)
    rows, cols = (x.astype(np.int32) for x in edges(pattern, n, m, rng))
    for drop, sym in ((False, False), (True, True)):
        g = bfs.Graph.from_coo_unique(n, rows, cols, drop_self_loops=drop, symmetrize=sym)
        off, cc = g.to_host()
        eoff, ecc = expected(n, rows, cols, drop, sym)
        assert np.array_equal(off, eoff)
        assert np.array_equal(cc, ecc)


@pytest.mark.parametrize("at", [0, 5000, 9999])
@pytest.mark.parametrize("row,col", [(100, 3), (3, 100), (-1, 3), (3, -(1 << 31))])
def test_id_out_of_range_is_named(at, row, col):
    rows, cols = np.arange(10000, dtype=np.int32) % 100, np.arange(10000, dtype=np.int32) % 97
    rows[at], cols[at] = row, col
    with pytest.raises(B40CError, match=r"edge %d \(%d,%d\) out of range \[0,100\)" % (at, row, col)):
        bfs.Graph.from_coo_unique(100, rows, cols, symmetrize=True)
