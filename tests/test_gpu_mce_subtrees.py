"""Subtrees of wide roots that are walked in registers: later neighbours over one to four words, earlier ones over up
to a dozen, cliques on both sides of 128 vertices, frames handed on from inside such a subtree.  Against the oracle;
whole numbers: no tolerance."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def graph_of(g2, m):
    a, b = np.nonzero(np.triu(m, 1))
    return g2.Graph.from_edges(a.astype(np.uint32), b.astype(np.uint32), len(m))


def hub(g2, x, p, dense, seed):
    """vertex x joined to x earlier and p later vertices, the later ones a random graph of that density"""
    rng = np.random.default_rng(seed)
    n = x + 1 + p
    m = np.zeros((n, n), bool)
    m[:x, :x] = rng.random((x, x)) < 0.05
    m[:x, x + 1:] = rng.random((x, p)) < 0.2
    m[x + 1:, x + 1:] = rng.random((p, p)) < dense
    m[:x, x] = True
    m[x, x + 1:] = True
    return graph_of(g2, m)


def cocktail(g2, n, pairs, before, seed):
    """K(n) without a matching of `pairs` edges (2^pairs cliques of n - pairs vertices), earlier vertices joined to
    random parts of it"""
    rng = np.random.default_rng(seed)
    m = np.zeros((before + n, before + n), bool)
    m[before:, before:] = True
    gone = before + rng.permutation(n)[:2 * pairs].reshape(pairs, 2)
    m[gone.min(1), gone.max(1)] = False
    m[:before, before:] = rng.random((before, n)) < 0.9
    return graph_of(g2, m)


def check(g2, orc, gpu_exec, g):
    every = np.arange(g.nv, dtype=np.uint32)
    with g2.Executor(device=0, mce_donate_every=1) as donating:
        for hist_len in (256, 70):
            ref = orc.mce(g, per_root=True, hist_len=hist_len)
            for ex in (gpu_exec, donating):
                ex.transfer(g)
                for kw in ({}, {"split": np.full(g.nv, 3, np.uint32)}, {"order": every[::-1].copy()}):
                    got = ex.run_mce(per_root=True, hist_len=hist_len, **kw)
                    assert got["total"] == ref["total"]
                    assert np.array_equal(got["hist"], ref["hist"])
                    assert np.array_equal(got["per_root_nodes"], ref["per_root_nodes"])


@pytest.mark.parametrize("x,p,dense", [(0, 65, 0.6), (63, 65, 0.6), (64, 100, 0.5), (300, 40, 0.5), (700, 60, 0.4),
                                       (200, 128, 0.4), (500, 129, 0.4), (40, 193, 0.3), (0, 257, 0.2), (4200, 30, 0.5)])
def test_wide_roots(g2, orc, gpu_exec, x, p, dense):
    print(f"case: {x} earlier, {p} later neighbours", flush=True)
    check(g2, orc, gpu_exec, hub(g2, x, p, dense, 1000 * x + p))


@pytest.mark.parametrize("n,pairs,before", [(70, 6, 0), (133, 6, 3), (135, 6, 20), (136, 5, 0), (200, 6, 70), (260, 4, 5)])
def test_large_cliques(g2, orc, gpu_exec, n, pairs, before):
    print(f"case: {n} vertices less {pairs} edges, {before} before them", flush=True)
    check(g2, orc, gpu_exec, cocktail(g2, n, pairs, before, n))
