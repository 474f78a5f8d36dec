"""Maximal cliques where the large-root pass takes more waves than the first
pass has: each of its waves needs a mailbox and a record area of its own.  Whole
numbers: equal to the oracle's, no tolerance."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def graph(g2, orc):
    g = g2.gen_chung_lu(3000, 2.3, 2.0, 400.0, 40_000, 11).preprocess().kcore_recode()[0]
    return g, orc.mce(g, per_root=True)


def check(got, ref):
    assert got["total"] == ref["total"]
    assert np.array_equal(got["hist"], ref["hist"])
    assert np.array_equal(got["per_root_nodes"], ref["per_root_nodes"])


@pytest.mark.parametrize("every", [1, 8])
def test_more_large_root_waves_than_first_pass_waves(g2, graph, every):
    """one wave per CU in the first pass, up to 2,048 in the large-root pass"""
    print("case: waves of the large-root pass, every", every, flush=True)
    g, ref = graph
    with g2.Executor(device=0, waves_per_cu=1, big_waves=2048, wave_scratch_words=64, mce_small_max=1,
                     mce_donate_every=every) as ex:
        ex.transfer(g)
        for _ in range(2):
            got = ex.run_mce(per_root=True)
            assert got["stats"]["big_roots"] > 256
            check(got, ref)


def dense_sides(g2, a, seed):
    """a random dense bipartite graph with a few edges within its sides, ids mixed"""
    rng = np.random.default_rng(seed)
    n = 2 * a
    m = np.zeros((n, n), bool)
    m[:a, a:] = rng.random((a, a)) < 0.9
    m[:a, :a] = rng.random((a, a)) < 0.01
    m[a:, a:] = rng.random((a, a)) < 0.01
    u, v = np.nonzero(np.triu(m, 1))
    ids = rng.permutation(n)
    return g2.Graph.from_edges(ids[u].astype(np.uint32), ids[v].astype(np.uint32), n)


def test_budgets_that_leave_few_waves(g2, orc):
    """the first pass shrinks to a few waves, and the large roots' arenas, for up
    to 256 waves, go to host memory"""
    print("case: waves of the large-root pass, budgets", flush=True)
    g = dense_sides(g2, 280, 3)
    ref = orc.mce(g, per_root=True)
    rows = sum((x + 255) // 256 * 256 for x in ((g.nv + 1) * 8, g.ne * 4, g.nv * 4, (g.nv + 1) * 4, (g.nv + 1) * 8))
    spilled = ran = 0
    for extra in (208, 224, 240, 440, 900, 3600):
        budget = rows + extra * 1024
        with g2.Executor(device=0, mem_budget=budget, wave_scratch_words=2048) as ex:
            ex.transfer(g)
            try:
                got = ex.run_mce(per_root=True)
            except RuntimeError as err:
                assert "(-3)" in str(err), (extra, err)  # G2_EBUDGET
                continue
        print("budget of", extra, "KiB beside the view:", got["stats"]["big_roots"], "large roots", flush=True)
        ran += 1
        spilled += got["stats"]["host_spill_bytes"] > 0
        assert got["stats"]["big_roots"] > 64
        assert got["stats"]["device_bytes"] <= budget
        check(got, ref)
    assert ran >= 4 and spilled >= 2
