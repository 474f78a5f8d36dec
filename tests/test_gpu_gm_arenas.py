"""Device memory of the counting walk's wave arenas.  Counts are whole numbers:
equal to the oracle's, no tolerance."""
import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def star(g2, d, chords, seed):
    """a hub joined to d vertices with a few edges among them"""
    rng = np.random.default_rng(seed)
    a, b = rng.integers(1, d + 1, (2, chords))
    src = np.concatenate((np.zeros(d, np.int64), a))
    dst = np.concatenate((np.arange(1, d + 1), b))
    keep = src != dst
    return g2.Graph.from_edges(src[keep].astype(np.uint32), dst[keep].astype(np.uint32), d + 1)


@pytest.mark.parametrize("d,q", [(9000, 0), (9000, 2), (5000, 7)])
def test_arenas_hold_the_stored_lists(g2, orc, d, q):
    """patterns of 3, 4 and 5 positions: no more memory than 16 waves per CU
    with two lists of the largest degree for every position (and 16 MB for the
    view, the windows and the counters)"""
    print("case: walk arenas", d, q, flush=True)
    g = star(g2, d, 300, 5)
    p = g2.plan_for_preset(q)
    ref = orc.gm(g, orc.OrcPlan.from_buffer_copy(bytes(p)), per_root=True)
    cus = importlib.import_module("g2-aimd_amd.device").device_info()["num_cus"]
    with g2.Executor(device=0) as ex:
        ex.transfer(g)
        ex.set_plan(p)
        got = ex.run_gm(per_root=True, canonical=True)
        solo = got["stats"]["device_bytes"]
        batch = ex.run_gm_batch([p])
    assert got["count"] == ref["count"] == batch["counts"][0]
    assert np.array_equal(got["per_root_count"], ref["per_root_count"])
    assert solo <= cus * 16 * d * 2 * p.n * 4 + (16 << 20)


def test_arena_of_one_list(g2, orc):
    """an edge: its only list, of rows within and beyond the LDS pool (1,280
    entries), alone and in a batch with patterns of 3 to 6 vertices"""
    print("case: walk arenas, an edge", flush=True)
    p = g2.plan_build([2, 1])
    others = [g2.plan_for_preset(q) for q in (0, 2, 7, 10)]
    for d in (1279, 1280, 1281, 4000):
        g = star(g2, d, 100, d)
        ref = orc.gm(g, orc.OrcPlan.from_buffer_copy(bytes(p)), per_root=True)
        assert ref["count"] == g.ne // 2
        with g2.Executor(device=0) as ex:
            ex.transfer(g)
            ex.set_plan(p)
            got = ex.run_gm(per_root=True, canonical=True)
            assert np.array_equal(got["per_root_count"], ref["per_root_count"]), d
            assert ex.run_gm_batch([p])["counts"].tolist() == [ref["count"]]
            counts = [orc.gm(g, orc.OrcPlan.from_buffer_copy(bytes(o)))["count"] for o in others]
            assert ex.run_gm_batch([others[0], p, *others[1:], p])["counts"].tolist() == \
                [counts[0], ref["count"], *counts[1:], ref["count"]]
