"""Maximal cliques of roots with more than 65,000 earlier neighbours, whose frames
take more than 1,022 words: they are handed on to idle waves too.  Whole numbers:
equal to the oracle's, no tolerance."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EARLIER = 66_000


@pytest.fixture(scope="module")
def case(g2, orc):
    """four hubs over the same earlier vertices; the first one's 40 later
    neighbours are joined at random, and every earlier vertex to two of them"""
    rng = np.random.default_rng(7)
    hubs = EARLIER + np.arange(4)
    first = EARLIER + 4 + np.arange(40)
    last = EARLIER + 44 + np.arange(6)
    x = np.arange(EARLIER)
    a, b = np.triu_indices(40, 1)
    keep = rng.random(len(a)) < 0.6
    two = rng.random((EARLIER, 40)).argsort(axis=1)[:, :2]
    src = [np.repeat(x, 4), np.repeat(x, 2), np.zeros(40, int) + hubs[0], first[a[keep]], np.repeat(hubs[1:], 2), last[::2]]
    dst = [np.tile(hubs, EARLIER), first[two].ravel(), first, first[b[keep]], last, last[1::2]]
    g = g2.Graph.from_edges(np.concatenate(src).astype(np.uint32), np.concatenate(dst).astype(np.uint32), EARLIER + 50)
    sources = hubs.astype(np.uint32)
    return g, sources, orc.mce(g, sources=sources, per_root=True)


@pytest.mark.parametrize("every", [1, 8])
def test_wide_frames_are_handed_on(g2, case, every):
    g, sources, ref = case
    print("case: wide frames, every", every, flush=True)
    with g2.Executor(device=0, mce_donate_every=every) as ex:
        ex.transfer(g, sources)
        got = ex.run_mce(per_root=True)
    print("nodes", ref["per_root_nodes"].tolist(), "donations", got["stats"]["donations"], flush=True)
    assert got["stats"]["big_roots"] == len(sources)
    assert got["total"] == ref["total"]
    assert np.array_equal(got["hist"], ref["hist"])
    assert np.array_equal(got["per_root_nodes"], ref["per_root_nodes"])
    assert got["stats"]["donations"] > 0
