"""The packed search on the GPU does hand work over: graphs with a few heavy
roots, of which thousands of waves have none of their own, give some away in
every mode, with the oracle's results."""
import numpy as np
import pytest

import rdmce_amd as R
from graphs import random_graph
from oracle_lib import OracleGraph, clique_hash

pytestmark = pytest.mark.gpu


def graph(kind):
    if kind == "skewed":
        g = R.Graph.rmat(11, 12, 0.57, 0.19, 0.19, seed=3)
    else:
        g = R.Graph.from_edges(random_graph(90, 0.7, 5))
    g.SortByOrder(R.OrderType.DEG)
    return g


@pytest.mark.parametrize("kind", ["skewed", "dense"])
@pytest.mark.parametrize("vertex,lists", [(False, False), (True, False), (False, True), (True, True)])
def test_work_is_given_away(kind, vertex, lists):
    print(f"[gpu-case] gifts {kind} vertex={vertex} lists={lists}", flush=True)
    g = graph(kind)
    og = OracleGraph.from_csr(g.GetRowOffset(), g.GetColIdx(), g.GetLabels(), g.GetDegeneracy())
    ref = og.mce(root_mode=1 if vertex else 2, root_nodes=True)
    p = R.Plan(g, pack=True, root_mode=R.ROOT_VERTEX if vertex else R.ROOT_EDGE, want_root_stats=True,
               want_list=lists, list_capacity=1 << 26 if lists else 0)
    given = 0
    for _ in range(3):
        out = p.run()
        assert (out.count, out.hash, out.hist_dict()) == (ref.count, ref.hash, ref.hist)
        assert np.array_equal(out.root_nodes, ref.root_nodes)
        if lists:
            assert len(out.cliques) == ref.count and clique_hash(out.cliques) == out.hash
        given += out.shared_tasks
    p.free()
    assert given > 0
