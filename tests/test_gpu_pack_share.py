"""The packed search handing work to idle waves: skewed graphs whose few heavy
roots and runs end up on many waves.  Bit-exact against the CPU oracle with
sharing on and off, with clique lists, root statistics and batches."""
import numpy as np
import pytest

import rdmce_amd as R
from graphs import dense_core_graph, random_graph
from oracle_lib import OracleGraph

pytestmark = pytest.mark.gpu


def oracle_for(g, root_mode=2, list_cap=0):
    og = OracleGraph.from_csr(g.GetRowOffset(), g.GetColIdx(), g.GetLabels(), g.GetDegeneracy())
    return og.mce(root_mode=root_mode, root_nodes=True, list_cap=list_cap)


def graph(kind):
    if kind == "rmat":       # runs of 90 roots, one- and two-word, X0' beyond 128
        g = R.Graph.rmat(12, 12, 0.57, 0.19, 0.19, seed=3)
    elif kind == "core":     # one dense core: all the work in a few runs
        g = R.Graph.from_edges(dense_core_graph(100, 4, 500, 0.02, 7))
    elif kind == "one word":  # |P0| <= 64: the first launch alone
        g = R.Graph.from_edges(random_graph(70, 0.7, 5))
    else:                    # below the sharing bound: nothing may be given away
        g = R.Graph.from_edges(random_graph(300, 0.05, 6))
    g.SortByOrder(R.OrderType.DEG)
    return g


@pytest.mark.parametrize("kind", ["rmat", "core", "one word", "sparse"])
@pytest.mark.parametrize("vertex,slots,share", [(False, 4, 0), (False, 1, 1), (True, 2, 0), (False, 4, -1)])
def test_shared_work_matches_oracle(kind, vertex, slots, share):
    print(f"[gpu-case] share {kind} vertex={vertex} slots={slots} share={share}", flush=True)
    g = graph(kind)
    mode = R.ROOT_VERTEX if vertex else R.ROOT_EDGE
    ref = oracle_for(g, 1 if vertex else 2, list_cap=1 << 22)
    lists = ref.count < 20000
    p = R.Plan(g, pack=True, pack_slots=slots, share_bound=share, root_mode=mode, want_root_stats=True,
               want_list=lists)
    for _ in range(3):  # who takes what differs from run to run
        out = p.run()
        assert (out.count, out.hash, out.hist_dict()) == (ref.count, ref.hash, ref.hist)
        assert out.total_nodes == ref.total_nodes
        assert np.array_equal(out.root_nodes, ref.root_nodes)
        if lists:
            assert sorted(out.cliques) == sorted(tuple(sorted(c)) for c in ref.cliques)
        if share < 0 or kind == "sparse" and share == 0:
            assert out.shared_tasks == 0
    p.free()
    plain = R.solve(g, root_mode=mode)
    assert out.search_bytes == plain.search_bytes


@pytest.mark.parametrize("replay", [False, True])
def test_shared_batch_matches_single_solves(replay):
    print(f"[gpu-case] share batch replay={replay}", flush=True)
    gs = [graph(k) for k in ("one word", "sparse", "core", "rmat")]
    b = R.Batch(gs, pack=True, use_graph=replay)
    refs = [oracle_for(g) for g in gs]
    for _ in range(3):
        out = b.run()
        for i, ref in enumerate(refs):
            assert (int(out.count[i]), int(out.hash[i]), out.hist_dict(i)) == (ref.count, ref.hash, ref.hist)
    b.free()
