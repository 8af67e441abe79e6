"""Several strategies in turn on one problem: what a search leaves in the
problem's counters is not read by the next one, whatever its strategy, form and
levels per host check."""
import numpy as np
import pytest

from helpers import csr_from_edges

pytestmark = pytest.mark.gpu

DEFAULT, ITERATIVE = 0, 2


def _path(n):
    return csr_from_edges(n, [(i, i + 1) for i in range(n - 1)], True)


@pytest.mark.parametrize("levels", [1, 2, 3, 6, 8])
@pytest.mark.parametrize("name", ["path5", "path9", "rmat12"])
def test_after_direction_optimizing(orc, name, levels):
    from back40computing_amd import _lib, bfs
    off, cols = orc.build_rmat_csr(12, 16, seed=3) if name == "rmat12" else _path(int(name[4:]))
    n = off.size - 1
    sources = [0, n // 2, n - 1] + ([int(s) for s in orc.pick_sources(off, 5, 3)] if name == "rmat12" else [])
    g = bfs.Graph.from_host_csr(off, cols)
    prob = bfs.CsrProblem()
    _lib.check(prob.FromGraph(g))
    first = bfs.ENACTORS[_lib.DIRECTION_OPTIMIZING]()
    first.set_tuning(levels_per_sync=levels)

    def search(en, src, mode, ref):
        _lib.check(prob.Reset(en.GetFrontierType(), 1.3))
        _lib.check(_lib.lib().b40c_enact_search(en.handle, prob.handle, src, 0, mode))
        depth, pred = prob.results()
        np.testing.assert_array_equal(depth, ref)
        assert orc.check_pred(off, cols, ref, pred) == -1
        assert en.GetStatistics()[1] == int(ref.max()) + 1

    for src in sources:
        ref = orc.bfs(off, cols, src, with_pred=False)[0]
        for strategy in sorted(bfs.ENACTORS):
            for mode in (ITERATIVE, DEFAULT):
                print("shared", name, levels, src, strategy, mode, flush=True)
                search(first, src, DEFAULT, ref)
                en = bfs.ENACTORS[strategy]()
                search(en, src, mode, ref)
                en.close()
    first.close()
    prob.close()
    g.close()
