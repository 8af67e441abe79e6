"""Batched results on both sides of the longest label array that is staged (2^18
words): staged alone, in windows, and copied, in turn and at random."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SCALES = [10, 18, 19]


@pytest.mark.parametrize("order", ["submitted", "shuffled"])
def test_stage_line(orc, order):
    from back40computing_amd import batch, bfs
    graphs = [bfs.Graph.rmat(s, 4, seed=s) for s in SCALES]
    host = [g.to_host() for g in graphs]
    mg = batch.MultiGraph(graphs)
    eng = batch.MultiSourceBFS(mg, 64 << 20, 32)
    queries = [(k % 3, int(s)) for k, s in enumerate(np.random.default_rng(5).integers(0, 1 << 10, 12))]
    ref = [orc.bfs(*host[g], s, with_pred=False)[0] for g, s in queries]
    for _ in range(2):
        ids = [eng.submit(g, s) for g, s in queries]
        eng.run()
        take = list(range(len(ids)))
        if order == "shuffled":
            np.random.default_rng(2).shuffle(take)
        for k, i in enumerate(take):
            print("stage line", order, queries[i], flush=True)
            g, s = queries[i]
            depth, pred, _ = eng.result(ids[i], g, want_pred=k % 3 != 0)
            assert np.array_equal(depth, ref[i])
            if k % 3:
                assert orc.check_pred(host[g][0], host[g][1], depth, pred) == -1
    eng.close()
    mg.close()
    for g in graphs:
        g.close()
