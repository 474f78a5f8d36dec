"""Matching at sizes few graphs reach: roots with more members than the hash index
holds on the general walker, and rows of 2^25 entries, with which the walk counts
its last position one candidate at a time.  Whole numbers: no tolerance."""
import numpy as np
import pytest

from test_gpu_gm_local import descending
from test_gpu_gm_wide import wide_graph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("a", [1040, 4097, 8190, 8191])
def test_wide_roots_general_walker(g2, gpu_exec, a):
    """three roots of K(a, a) with a graph of 24 vertices in its second side, the
    plans' symmetry breaking reversed so that they are no clique plans"""
    print("case: wide roots, general walker", a, flush=True)
    g, cliques = wide_graph(g2, a, a)
    gpu_exec.transfer(g, np.array([0, a // 2, a - 1], np.uint32))
    for q, n in ((0, 3), (24, 4), (25, 5)):
        print("  cliques of", n, flush=True)
        plan = descending(g2, g2.plan_for_preset(q))
        assert g2.plan_local_eligible(plan)
        gpu_exec.set_plan(plan)
        r = gpu_exec.run_gm()
        assert r["stats"]["local_bitmap"] == 1 and r["stats"]["local_pass_roots"][4] == 3
        assert r["count"] == 3 * cliques[n - 1]


@pytest.mark.parametrize("d", [(1 << 25) - 1, 1 << 25])
def test_rows_of_2_to_25_entries(g2, orc, d):
    """vertex 2 is joined to all d others, seven of which form a clique"""
    print("case: walk, a row of", d, "entries", flush=True)
    clique = np.array([0, 1, 5, 6, 7, 70, d], np.int64)
    deg = np.ones(d + 1, np.int64)
    deg[clique] = len(clique)
    deg[2] = d
    rp = np.concatenate(([0], np.cumsum(deg)))
    cols = np.full(rp[-1], 2, np.uint32)
    cols[rp[2]:rp[3]] = np.delete(np.arange(d + 1, dtype=np.uint32), 2)
    for v in clique:
        cols[rp[v]:rp[v + 1]] = np.sort(np.append(clique[clique != v], 2))
    g = g2.Graph(rp.astype(np.uint64), cols)
    sources = np.array([0, 1, 5, 70, 1000], np.uint32)
    with g2.Executor(device=0, mem_budget=4 << 30, block_waves=1, waves_per_cu=1) as ex:
        ex.transfer(g, sources)
        for q in (0, 2, 24):
            p = g2.plan_for_preset(q)
            ex.set_plan(p)
            ref = orc.gm(g, orc.OrcPlan.from_buffer_copy(bytes(p)), sources=sources, per_root=True)
            got = ex.run_gm(per_root=True, canonical=True)
            assert ref["count"] > 0 and got["count"] == ref["count"], q
            assert np.array_equal(got["per_root_count"], ref["per_root_count"]), q
            assert ex.run_gm_batch([p])["counts"].tolist() == [ref["count"]], q
