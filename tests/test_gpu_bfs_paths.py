"""Searches at the sizes where the gather and claim paths change: graphs on
both sides of the label-claim limit, tiles dealt out in every turn length,
frontier pieces that overflow into the shared queue, hub lists split over
workgroups, bottom-up levels followed by top-down ones, wide contractions, and
directed graphs whose deepest vertices have no out-edges.  Depths and search
depth are compared exactly with the serial oracle, predecessors with the
search's invariants."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EC, CE, TP, HYBRID, DO = 0, 1, 2, 3, 5
DEFAULT, FUSED, ITERATIVE = 0, 1, 2
FORMS = [(EC, FUSED), (EC, ITERATIVE), (CE, FUSED), (CE, ITERATIVE), (TP, FUSED), (TP, ITERATIVE), (HYBRID, DEFAULT),
         (DO, DEFAULT)]


def _csr(n, rows, cols, undirected=True):
    r = np.concatenate([rows, cols]) if undirected else np.asarray(rows)
    c = np.concatenate([cols, rows]) if undirected else np.asarray(cols)
    key = np.unique(r.astype(np.int64) * n + c)
    off = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(key // n, minlength=n), out=off[1:])
    return off.astype(np.int32), (key % n).astype(np.int32)


def _star(leaves):
    # A hub, its leaves, and a tail behind the last leaf.
    n = leaves + 4
    rows = np.concatenate([np.zeros(leaves, np.int64), [leaves, leaves + 1, leaves + 2]])
    cols = np.concatenate([np.arange(1, leaves + 1), [leaves + 1, leaves + 2, leaves + 3]])
    return _csr(n, rows, cols)


def _sparse(n, degree, seed):
    rng = np.random.default_rng(seed)
    m = n * degree // 2
    return _csr(n, rng.integers(0, n, m), rng.integers(0, n, m))


def _sinks(n, seed):
    # Layers of out-edges only; the last layer has none.
    rng = np.random.default_rng(seed)
    layer = np.sort(rng.integers(0, 6, n))
    layer[0] = 0
    rows = rng.integers(0, n, 8 * n)
    cols = rng.integers(0, n, 8 * n)
    keep = layer[cols] == layer[rows] + 1
    return _csr(n, rows[keep], cols[keep], undirected=False)


def _hubs(n, seed):
    # Several hubs of different degrees over a sparse graph.
    rng = np.random.default_rng(seed)
    rows = [rng.integers(0, n, n)]
    cols = [rng.integers(0, n, n)]
    for hub, deg in ((1, 255), (2, 256), (3, 2047), (4, 2048), (5, n // 3), (6, n // 2)):
        rows.append(np.full(deg, hub))
        cols.append(rng.integers(0, n, deg))
    return _csr(n, np.concatenate(rows), np.concatenate(cols))


GRAPHS = {
    "star_300": lambda: _star(300),
    "star_spill": lambda: _star(1_100_000),
    "sparse_label": lambda: _sparse(1 << 20, 6, 1),
    "sparse_bitmask": lambda: _sparse((1 << 20) + 1, 6, 2),
    "sparse_small": lambda: _sparse(4095, 5, 3),
    "sinks": lambda: _sinks(60_000, 4),
    "hubs": lambda: _hubs(150_000, 5),
}


@pytest.mark.parametrize("name", sorted(GRAPHS))
def test_paths_against_oracle(orc, name):
    from back40computing_amd import autotune, bfs
    off, cols = GRAPHS[name]()
    g = bfs.Graph.from_host_csr(off, cols)
    edge_keys = autotune.sorted_edge_keys(off, cols)
    sources = [0, int(np.argmax(np.diff(off)))]
    if name.startswith("star"):
        sources.append(off.size - 2)
    for src in sorted(set(sources)):
        ref = orc.bfs(off, cols, src, with_pred=False)[0]
        for strategy, mode in FORMS:
            for tuning in (None, {"grid_gather_threshold": 64, "do_alpha": 1000, "do_beta": 2},
                           {"grid_gather_threshold": 1 << 30, "grid_size": 7, "persistent_wgs_per_cu": 1}):
                if tuning and off.size > 200_000 and (strategy, mode) not in FORMS[:2] + FORMS[-1:]:
                    continue
                print("paths", name, src, strategy, mode, tuning, flush=True)
                depth, pred, st = bfs.bfs(g, src, strategy=strategy, mode=mode, tuning=tuning)
                np.testing.assert_array_equal(depth, ref)
                assert autotune.verify_bfs_labels(off, cols, src, depth, pred, edge_keys, depth_verified=True)
                assert st["search_depth"] == int(ref.max()) + 1
    g.close()


@pytest.mark.parametrize("edges", [(1 << 19) - 2, 1 << 19])
def test_default_grid_tier_line(orc, edges):
    """Both sides of the number of edges from which lists of 128 edges go to
    the grid tier, with lists of 127, 128 and 129 edges and a few longer ones."""
    from back40computing_amd import autotune, bfs
    rng = np.random.default_rng(edges)
    n = 6000
    deg = np.concatenate([[400, 127, 128, 129, 2047, 2048, 2049, 5000], rng.choice([0, 1, 60, 127, 128, 129], n)])
    deg = np.concatenate([deg, np.full(n, (edges - int(deg.sum())) // n)])
    deg[-1] += edges - int(deg.sum())
    off = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    assert off[-1] == edges
    cols = rng.integers(0, deg.size, edges).astype(np.int32)
    g = bfs.Graph.from_host_csr(off, cols)
    edge_keys = autotune.sorted_edge_keys(off, cols)
    ref = orc.bfs(off, cols, 0, with_pred=False)[0]
    for strategy, mode in FORMS:
        print("grid tier line", edges, strategy, mode, flush=True)
        depth, pred, st = bfs.bfs(g, 0, strategy=strategy, mode=mode)
        np.testing.assert_array_equal(depth, ref)
        assert autotune.verify_bfs_labels(off, cols, 0, depth, pred, edge_keys, depth_verified=True)
    g.close()
