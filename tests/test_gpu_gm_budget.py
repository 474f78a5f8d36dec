"""The node budget of batched matching on a query whose walks end before their
last position: node counts are whole numbers, bounds are exact."""
import pytest

import graphs as G

pytestmark = pytest.mark.gpu


def test_budget_stops_walks_without_matches(g2, gpu_exec):
    """an odd cycle with two pendant vertices in a complete bipartite graph: the
    cycle never closes, at the position before the last.  Each wave may charge a
    block of nodes and one list (of at most 30) before it sees the limit passed"""
    print("case: node budget, no last position", flush=True)
    query = [0] * 7
    for a, b in ((0, 1), (1, 2), (2, 3), (3, 4), (4, 0), (0, 5), (2, 6)):
        query[a] |= 1 << b
        query[b] |= 1 << a
    p = g2.plan_build(query)
    last = p.n - 1
    assert list(p.bn[last - 1][:p.bn_count[last - 1]]) == [2, 4]  # the cycle's closing
    gpu_exec.transfer(G.complete_bipartite(g2, 30, 30))
    whole = gpu_exec.run_gm_batch([p])
    assert whole["counts"].tolist() == [0] and not whole["over_budget"].any()
    limit, waves = 100_000, 16 * 256
    bound = limit + waves * (2 * 256 + 30)
    assert whole["nodes"][0] > 4 * bound
    got = gpu_exec.run_gm_batch([p], node_budget=limit)
    assert got["over_budget"].tolist() == [True]
    assert limit < got["nodes"][0] <= bound
