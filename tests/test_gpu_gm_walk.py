"""The counting walk (per-root counts, patterns that are no cliques, batches)
at the sizes where its routes change: row lengths around the window bounds of
3, 4 and 5 positions and around the LDS list pool, sources that repeat, runs of
sources, and a budget too small for the list of windows.  Counts are whole
numbers: equal to the oracle's, no tolerance."""
import numpy as np
import pytest

import graphs as G

pytestmark = pytest.mark.gpu


def hubs(g2, d, seed=1):
    """two joined hubs over the same d vertices, which form a cycle with a few
    chords: every hub pair's common row is d long, the other rows are short"""
    rng = np.random.default_rng(seed)
    v = np.arange(2, d + 2)
    chords = rng.integers(2, d + 2, (2, max(1, d // 16)))
    src = np.concatenate(([0], np.zeros(d, int), np.ones(d, int), v, chords[0]))
    dst = np.concatenate(([1], v, v, np.roll(v, 1), chords[1]))
    keep = src != dst
    return g2.Graph.from_edges(src[keep].astype(np.uint32), dst[keep].astype(np.uint32), d + 2)


def check(g2, orc, ex, g, q, sources=None):
    p = g2.plan_for_preset(q)
    ex.transfer(g, sources)
    ex.set_plan(p)
    got = ex.run_gm(per_root=True, canonical=True)
    ref = orc.gm(g, orc.OrcPlan.from_buffer_copy(bytes(p)), sources=sources, per_root=True)
    assert got["count"] == ref["count"], (q, got["count"], ref["count"])
    assert np.array_equal(got["per_root_count"], ref["per_root_count"]), q
    # the extensions the accounting traversal counts are the walk's
    assert got["stats"]["nodes"] == ex.run_gm(account=True)["stats"]["nodes"], q
    batch = ex.run_gm_batch([p, p])
    assert batch["counts"].tolist() == [ref["count"]] * 2
    assert batch["nodes"].tolist() == [got["stats"]["nodes"]] * 2


@pytest.mark.parametrize("d", [1, 7, 8, 9, 63, 64, 65, 127, 128, 129])
def test_row_lengths_all_sizes(g2, orc, gpu_exec, d):
    print("case: walk, hub rows of", d, flush=True)
    for q in (0, 1, 2, 5, 7, 16, 24):
        check(g2, orc, gpu_exec, hubs(g2, d), q)


@pytest.mark.parametrize("d", [255, 256, 511, 513, 1023, 1025, 1279, 1281, 2600])
def test_row_lengths_pool(g2, orc, gpu_exec, d):
    """lists that just fit, or do not fit, the LDS pool; 3 and 4 positions
    (and 5 where the hubs' matches stay few)"""
    print("case: walk, hub rows of", d, flush=True)
    for q in (0, 1, 2, 24, 25):
        check(g2, orc, gpu_exec, hubs(g2, d), q)


@pytest.mark.parametrize("d", [9, 65, 400])
def test_batch_of_mixed_sizes(g2, orc, gpu_exec, d):
    """one list of windows serves plans of 3 to 5 positions"""
    print("case: walk, mixed batch, hub rows of", d, flush=True)
    g = hubs(g2, d)
    plans = [g2.plan_for_preset(q) for q in (5, 0, 24, 2, 1, 5, 23)]
    gpu_exec.transfer(g)
    got = gpu_exec.run_gm_batch(plans, order=np.arange(len(plans))[::-1])
    ref = [orc.gm(g, orc.OrcPlan.from_buffer_copy(bytes(p)))["count"] for p in plans]
    assert got["counts"].tolist() == ref


def test_sources(g2, orc, gpu_exec):
    """sources in any order and repeated, and more sources than a block of them"""
    print("case: walk, sources", flush=True)
    g = hubs(g2, 200)
    rng = np.random.default_rng(3)
    for s in (np.array([0], np.uint32), np.array([5, 0, 5, 1, 0], np.uint32), rng.permutation(g.nv).astype(np.uint32)):
        for q in (2, 5):
            check(g2, orc, gpu_exec, g, q, s)
    many = G.gnp(g2, 3000, 0.004, 2)
    s = rng.integers(0, many.nv, 200_000).astype(np.uint32)
    p = g2.plan_for_preset(2)
    gpu_exec.transfer(many, s)
    gpu_exec.set_plan(p)
    got = gpu_exec.run_gm(per_root=True)["per_root_count"]
    gpu_exec.transfer(many)
    assert np.array_equal(got, gpu_exec.run_gm(per_root=True)["per_root_count"][s])


def test_budget_without_window_list(g2, orc):
    """a budget that holds the view and one workgroup's lists but no list of
    windows: the rows are walked whole"""
    print("case: walk, no room for the windows", flush=True)
    g = hubs(g2, 513)
    p = g2.plan_for_preset(5)
    ref = orc.gm(g, orc.OrcPlan.from_buffer_copy(bytes(p)), per_root=True)
    with g2.Executor(device=0, mem_budget=4 * 514 * 2 * p.n * 4 + 60_000) as ex:
        ex.transfer(g)
        ex.set_plan(p)
        got = ex.run_gm(per_root=True)
    assert got["count"] == ref["count"]
    assert np.array_equal(got["per_root_count"], ref["per_root_count"])
