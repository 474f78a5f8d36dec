"""The list of the long root rows' windows: its size where single entries are
dealt out in 8, 4, 2 and 1 parts and where windows hold several entries, and its
room under a budget, which other buffers come before.  Counts are whole numbers:
equal to the oracle's, no tolerance."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MB = 1 << 20


def bipartite(g2, a):
    """complete bipartite graph with a triangle on one side: every entry joins
    two rows of a vertices, so that every window is dealt out in the most parts"""
    u, v = np.repeat(np.arange(a), a), np.tile(a + np.arange(a), a)
    return g2.Graph.from_edges(np.concatenate((u, [0, 0, 1])).astype(np.uint32),
                               np.concatenate((v, [1, 2, 2])).astype(np.uint32), 2 * a)


def sparse(g2, nv, edges, hub, seed):
    """random graph with two joined hubs over `hub` vertices and a clique of 30"""
    rng = np.random.default_rng(seed)
    e = rng.integers(0, nv, (2, edges))
    few = rng.permutation(np.arange(2, nv))
    a, b = np.triu_indices(30, 1)
    src = np.concatenate((e[0], [0], np.zeros(hub, np.int64), np.ones(hub, np.int64), few[a]))
    dst = np.concatenate((e[1], [1], few[:hub], few[:hub], few[b]))
    keep = src != dst
    return g2.Graph.from_edges(src[keep].astype(np.uint32), dst[keep].astype(np.uint32), nv)


GRAPHS = {
    # row entries: 101k (room for 8 parts everywhere), 500k to 2M (8 parts by the degrees), 2.9M, 3.9M (4 parts)
    "k225": lambda g2: bipartite(g2, 225), "k500": lambda g2: bipartite(g2, 500), "k700": lambda g2: bipartite(g2, 700),
    "k1000": lambda g2: bipartite(g2, 1000), "k1200": lambda g2: bipartite(g2, 1200),
    "k1400": lambda g2: bipartite(g2, 1400),
    # 3.0M and 5.2M row entries: windows of one entry, of two
    "sparse1": lambda g2: sparse(g2, 60_000, 1_500_000, 3000, 1), "sparse2": lambda g2: sparse(g2, 100_000, 2_600_000, 3000, 2),
}


@pytest.mark.parametrize("name,q", [(n, 8) for n in GRAPHS] + [("sparse1", 5), ("sparse2", 5)])
def test_list_is_bounded(g2, orc, name, q):
    """5 positions: room for at most 8 parts of every window, by the degrees, and
    at most 2^24 windows; the counts of the walk (alone, per root, in a batch, with
    a caller's windows) are the oracle's"""
    g = GRAPHS[name](g2)
    print("case: windows", name, g.ne, "row entries, pattern", q, flush=True)
    p = g2.plan_for_preset(q)
    ref = orc.gm(g, orc.OrcPlan.from_buffer_copy(bytes(p)), per_root=True)
    with g2.Executor(device=0, waves_per_cu=2) as ex:
        ex.transfer(g)
        ex.set_plan(p)
        got = ex.run_gm(per_root=True, canonical=True)
        assert got["count"] == ref["count"]
        assert np.array_equal(got["per_root_count"], ref["per_root_count"])
        # row offsets, degrees, sources, window offsets, per-root counts; columns; arenas of 6 lists
        rest = 40 * g.nv + 4 * g.ne + 256 * 2 * int(g.degrees().max()) * 6 * 4 + 5 * MB
        d = g.degrees().astype(np.int64)
        most = 9 * g.ne if g.ne <= 466_000 else min(1 << 24, max((d * np.minimum(8, 1 + d // 32)).sum(), g.ne + g.ne // 8))
        assert got["stats"]["device_bytes"] - rest <= 16 * most
        for window in (0, 1):
            assert ex.run_gm_batch([p], window=window)["counts"].tolist() == [ref["count"]]


def test_list_gives_way(g2, orc):
    """a budget that holds a run's list exactly: the repeated run has it again, a
    larger view is taken afterwards, and other runs find the list's room"""
    print("case: windows give way", flush=True)
    small, large = sparse(g2, 40_000, 700_000, 2000, 3), sparse(g2, 40_000, 1_400_000, 2000, 4)
    p, tri = g2.plan_for_preset(8), g2.plan_for_preset(0)
    tune = dict(waves_per_cu=2, wave_scratch_words=4096)
    count = [orc.gm(g, orc.OrcPlan.from_buffer_copy(bytes(p)))["count"] for g in (small, large)]
    with g2.Executor(device=0, **tune) as ex:
        ex.transfer(small)
        ex.set_plan(p)
        held = ex.run_gm(canonical=True)["stats"]["device_bytes"]
    with g2.Executor(device=0, mem_budget=held, **tune) as ex:
        ex.transfer(small)
        ex.set_plan(p)
        for _ in range(2):
            got = ex.run_gm(canonical=True)
            assert got["count"] == count[0] and got["stats"]["device_bytes"] == held
        ex.transfer(large)
        assert ex.run_gm(canonical=True)["count"] == count[1]
        ex.set_plan(tri)
        ref = orc.gm(large, orc.OrcPlan.from_buffer_copy(bytes(tri)))
        assert ex.run_gm(account=True)["count"] == ref["count"]
        got, ref = ex.run_mce(), orc.mce(large)
        assert got["total"] == ref["total"] and np.array_equal(got["hist"], ref["hist"])
