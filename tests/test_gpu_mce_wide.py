"""Maximal cliques of roots with up to 64 later neighbours whose earlier ones
take several words: the walk that keeps those words in registers, at the word
bounds and on both sides of its limits, against the oracle.  Whole numbers: no
tolerance."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def hub(g2, x, p, seed):
    """Vertex x is joined to all of 0 .. x - 1 and of x + 1 .. x + p; every
    earlier vertex has a later neighbour, so |X'| of root x is x."""
    rng = np.random.default_rng(seed)
    n = x + 1 + p
    m = np.zeros((n, n), bool)
    m[:x, :x] = rng.random((x, x)) < 0.05
    m[:x, x + 1:] = rng.random((x, p)) < 0.3
    m[np.arange(x), x + 1 + np.arange(x) % p] = True
    m[x + 1:, x + 1:] = rng.random((p, p)) < 0.7
    m[:x, x] = True
    m[x, x + 1:] = True
    a, b = np.nonzero(np.triu(m, 1))
    return g2.Graph.from_edges(a.astype(np.uint32), b.astype(np.uint32), n)


@pytest.mark.parametrize("x,p", [(1, 64), (64, 1), (64, 40), (65, 40), (128, 40), (129, 63), (192, 30), (256, 64),
                                 (257, 40), (256, 65), (300, 2)])
def test_register_walk_limits(g2, orc, gpu_exec, x, p):
    print(f"case: {x} earlier, {p} later neighbours", flush=True)
    g = hub(g2, x, p, 100 * x + p)
    ref = orc.mce(g, per_root=True)
    every = np.arange(g.nv, dtype=np.uint32)
    with g2.Executor(device=0, mce_donate_every=1) as donating:
        for ex in (gpu_exec, donating):
            ex.transfer(g)
            for kw in ({}, {"split": np.full(g.nv, 5, np.uint32)}, {"order": every[::-1].copy()}):
                got = ex.run_mce(per_root=True, **kw)
                assert got["total"] == ref["total"]
                assert np.array_equal(got["hist"], ref["hist"])
                assert np.array_equal(got["per_root_nodes"], ref["per_root_nodes"])
