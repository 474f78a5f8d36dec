"""Root features at the sizes where the kernels change their split: rows of 16
and 64 neighbours (the sketch maxima), roots of 149 and 1040 members (the
triangle counts' indexes).  Whole numbers with a closed form, the 2-hop
estimate from the oracle: no tolerance."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(2, 3, 16, 17, 18, 64, 65, 66, 128, 129, 130), (149, 150, 151, 152, 5), (1040, 1041, 1042, 1043)])
def test_cliques_of_every_split(g2, gpu_exec, sizes):
    """Disjoint cliques with a pendant vertex each: every clique vertex lies on
    all of its clique's triangles, its pendant on none."""
    print("case: features of cliques", sizes, flush=True)
    pairs, feats, at = [], [], 0
    for k in sizes:
        i, j = np.triu_indices(k, 1)
        pairs.append(np.stack([i + at, j + at]))
        pairs.append(np.array([[at + k - 1], [at + k]]))
        for v in range(k):
            feats.append((k - 1 + (v == k - 1), (k - 1) * (k - 2) // 2, k - 1 if k > 2 else 0, max(k - 1 - v, 1)))
        feats.append((1, 0, 0, 0))
        at += k + 1
    e = np.concatenate(pairs, axis=1).astype(np.uint32)
    g = g2.Graph.from_edges(e[0], e[1], at)
    gpu_exec.transfer(g)
    f = gpu_exec.features()
    assert np.array_equal(f[:, [0, 2, 3, 4]], np.array(feats, np.int64))
    assert np.array_equal(f[:, 1], oracle.two_hop(g))
    src = np.arange(1, g.nv, 3, dtype=np.uint32)
    gpu_exec.transfer(g2.view_materialize(g, src, 2), sources=src)
    assert np.array_equal(gpu_exec.features(), f[src])
