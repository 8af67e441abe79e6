"""Batched search where its push and its counts change form: hubs around the grid
tier's threshold and beyond one gather step, few and many queries per graph, and
more (graph, slot) pairs in a level than the counts' table holds."""
import numpy as np
import pytest

from helpers import csr_from_edges

pytestmark = pytest.mark.gpu


def _hubs(n, degrees, seed):
    """A ring with chords from the first vertices, of the given degrees."""
    rng = np.random.default_rng(seed)
    edges = [(i, (i + 1) % n) for i in range(n)]
    for h, d in enumerate(degrees):
        edges += [(h, int(x)) for x in rng.choice(n, min(d, n - 1), replace=False) if int(x) != h]
    return csr_from_edges(n, edges, True)


@pytest.mark.parametrize("graphs,per_graph", [(1, 1), (1, 64), (3, 16), (3, 17), (40, 15), (40, 33)])
@pytest.mark.parametrize("lps", [0, 4, -2])
def test_hubs_and_slots(orc, graphs, per_graph, lps):
    from back40computing_amd import batch, bfs
    kinds = [(1500, [127, 128, 129, 255, 256, 257, 1200]), (6000, [5900, 1023, 1025]), (97, [50]), (700, [])]
    host = [_hubs(n, d, k) for k, (n, d) in enumerate(kinds)]
    pool = [bfs.Graph.from_host_csr(o, c) for o, c in host]
    mg = batch.MultiGraph([pool[g % 4] for g in range(graphs)])
    eng = batch.MultiSourceBFS(mg, label_budget_bytes=1 << 28)
    if lps < 0:
        eng.set_persistent(True)
    eng.set_levels_per_step(abs(lps))
    rng = np.random.default_rng(graphs * 100 + per_graph)
    queries = [(g, int(s)) for g in range(graphs) for s in rng.integers(0, mg.nodes(g), per_graph)]
    ids = [eng.submit(g, s) for g, s in queries]
    eng.run()
    ref = {}
    for q, (g, s) in zip(ids, queries):
        if (g % 4, s) not in ref:
            ref[g % 4, s] = orc.bfs(*host[g % 4], s, with_pred=False)
        depth, pred, levels = eng.result(q, g)
        want, _, want_levels = ref[g % 4, s]
        assert np.array_equal(depth, want)
        assert levels == want_levels
        assert orc.check_pred(*host[g % 4], want, pred) == -1
    eng.close()
    mg.close()
