"""Results of a batch taken in every order: labels pass through a stage that holds
several queries' labels, so each order, mix of wanted labels, early release and
reuse of ids and label memory has to give each query its own."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SCALES = [6, 9, 12, 18]  # the last one's labels are too long for the stage
PER_GRAPH = 40


@pytest.fixture(scope="module")
def pool():
    from back40computing_amd import batch, bfs
    graphs = [bfs.Graph.rmat(s, 8, seed=s) for s in SCALES]
    host = [g.to_host() for g in graphs]
    return batch.MultiGraph(graphs), host


@pytest.mark.parametrize("order", ["submitted", "reversed", "shuffled", "alternate", "pairs_swapped"])
def test_result_orders(pool, orc, order):
    from back40computing_amd import batch
    mg, host = pool
    rng = np.random.default_rng(len(order))
    per = [PER_GRAPH, PER_GRAPH, PER_GRAPH, 3]
    queries = [(g, int(s)) for g in range(len(SCALES)) for s in orc.pick_sources(host[g][0], 7 + g, per[g])]
    words = sum(mg.nodes(g) for g, _ in queries)
    eng = batch.MultiSourceBFS(mg, int(words * 8 * 1.1), len(queries) + 4)
    want_depth = {}
    for g, s in queries:
        if (g, s) not in want_depth:
            want_depth[g, s] = orc.bfs(*host[g], s, with_pred=False)[0]
    for _ in range(2):  # the second time with recycled ids and label memory
        rng.shuffle(queries)
        ids = [eng.submit(g, s) for g, s in queries]
        eng.run()
        take = list(range(len(ids)))
        if order == "reversed":
            take.reverse()
        elif order == "shuffled":
            rng.shuffle(take)
        elif order == "pairs_swapped":
            take = [i ^ 1 if (i ^ 1) < len(ids) else i for i in take]
        for k, i in enumerate(take):
            g, s = queries[i]
            if order == "alternate" and k % 5 == 3:
                eng.release(ids[i])
                continue
            pred_too = order in ("submitted", "shuffled") or k % 2 == 0
            depth, pred, levels = eng.result(ids[i], g, want_pred=pred_too)
            assert np.array_equal(depth, want_depth[g, s])
            assert levels == depth.max() + 1
            if pred_too:
                assert orc.check_pred(host[g][0], host[g][1], depth, pred) == -1
            if k == len(take) // 2:  # a query in between, while others are staged
                q = eng.submit(0, queries[0][1] % mg.nodes(0))
                eng.run()
                eng.release(q)
