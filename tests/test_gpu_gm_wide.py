"""Roots too large for a workgroup's LDS (|U| >= 1040), at the sizes where their kernels change: the first one, more
than 64 words a row, and on both sides of the hash index's capacity.  Counts have a closed form: no tolerance."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def wide_graph(g2, a, seed):
    """K(a, a) with a random graph of 24 vertices placed into its second side, ends included: each of the first a
    vertices is the lowest of U = the second side, |U| = a.  Returns it with the cliques of 2 .. 5 in that graph."""
    rng = np.random.default_rng(seed)
    k = 24
    place = np.sort(np.concatenate(([0, a - 1], rng.choice(np.arange(1, a - 1), k - 2, replace=False))))
    adj = np.triu(rng.random((k, k)) < 0.6, 1)
    cliques = {1: [(i,) for i in range(k)]}
    for n in range(2, 6):
        cliques[n] = [c + (j,) for c in cliques[n - 1] for j in range(c[-1] + 1, k) if all(adj[i, j] for i in c)]
    adj = adj | adj.T
    side_a, side_b = np.arange(a, dtype=np.uint32), np.arange(a, 2 * a, dtype=np.uint32)
    rows = [np.tile(side_b, a)]
    deg = np.full(2 * a, a, np.uint64)
    at = 0
    for i, p in enumerate(place):
        rows += [np.tile(side_a, p - at), side_a, (a + place[adj[i]]).astype(np.uint32)]
        deg[a + p] += int(adj[i].sum())
        at = p + 1
    rows.append(np.tile(side_a, a - at))
    rp = np.concatenate(([0], np.cumsum(deg))).astype(np.uint64)
    return g2.Graph(rp, np.concatenate(rows)), {n: len(c) for n, c in cliques.items()}


@pytest.mark.parametrize("a", [1040, 1049, 4100, 8191])
def test_wide_roots(g2, gpu_exec, a):
    print("case: wide roots", a, flush=True)
    g, cliques = wide_graph(g2, a, a)
    gpu_exec.transfer(g)
    for q, n in ((0, 3), (24, 4), (25, 5)):
        print("  cliques of", n, flush=True)
        gpu_exec.set_plan(g2.plan_for_preset(q))
        r = gpu_exec.run_gm()
        assert r["stats"]["local_pass_roots"][4] == a
        assert r["count"] == a * cliques[n - 1] + cliques[n]
