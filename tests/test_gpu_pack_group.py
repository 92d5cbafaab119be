"""The bitmap of a vertex run in the packed search: its lower neighbours' rows
are built for all of them, and those without a bit are dropped by moving the
others together.  Runs whose sets end at, before and after a 64 boundary, with
no, some and only non-empty rows, bit-exact against the CPU oracle."""
import numpy as np
import pytest

import rdmce_amd as R
from oracle_lib import OracleGraph

pytestmark = pytest.mark.gpu


def run_graph(d0, seed):
    """Vertices with d0 later neighbours U (random, joined to a clique so that
    they come later in the order) and x0 earlier ones, each of which has 1 to 3
    neighbours in U with probability `keep`, else none."""
    rng = np.random.default_rng(seed)
    edges = [(i, j) for i in range(d0) for j in range(i + 1, d0) if rng.random() < 0.4]
    w = range(d0, d0 + d0 + 3)
    edges += [(i, j) for i in w for j in w if i < j]
    edges += [(i, j) for i in range(d0) for j in w]
    n = 2 * d0 + 3
    for x0 in (0, 1, 63, 64, 65, 130, 200):
        for keep in (0.0, 0.5, 1.0):
            v = n
            n += 1
            edges += [(v, u) for u in range(d0)]
            for _ in range(x0):
                edges.append((v, n))
                if rng.random() < keep:
                    edges += [(n, int(u)) for u in rng.choice(d0, rng.integers(1, 4), replace=False)]
                n += 1
    return R.Graph.from_edges(np.array(edges))


@pytest.mark.parametrize("d0", [5, 63, 64, 65, 127, 130])
def test_runs_at_word_edges(d0):
    print(f"[gpu-case] run bitmaps d0={d0}", flush=True)
    g = run_graph(d0, 3)
    g.SortByOrder(R.OrderType.DEG)
    og = OracleGraph.from_csr(g.GetRowOffset(), g.GetColIdx(), g.GetLabels(), g.GetDegeneracy())
    ref = og.mce(root_mode=2, root_nodes=True)
    p = R.Plan(g, pack=True, want_root_stats=True)
    for _ in range(2):
        out = p.run()
        assert (out.count, out.hash, out.hist_dict()) == (ref.count, ref.hash, ref.hist)
        assert np.array_equal(out.root_nodes, ref.root_nodes)
    p.free()
