"""The local-bitmap passes' hash index over a root's members (lookups of
streamed row entries) where its slots hold chains.  Counts are whole numbers
with a closed form: no tolerance."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("stride,size", [(512, 60), (512, 149), (8192, 40), (1024, 151), (1024, 156)])
def test_members_that_share_hash_slots(g2, gpu_exec, stride, size):
    """Disjoint cliques on the vertices j, j + stride, j + 2 stride, ..: all
    degrees are equal, so rank is id, and a root's members share one slot of
    the wave's index (stride 512, 8192: with equal tags) or a few of the
    workgroup's (stride 1024).  Roots on both sides of the wave's limit of 149
    members.  k-cliques are stride x C(size, k)."""
    print(f"case: members sharing hash slots, stride {stride}, size {size}", flush=True)
    n = stride * size
    k = np.arange(size - 1, dtype=np.uint32)
    own = np.arange(n, dtype=np.uint32) // stride
    cols = (k + (k >= own[:, None])) * np.uint32(stride) + np.arange(n, dtype=np.uint32)[:, None] % np.uint32(stride)
    g = g2.Graph(np.arange(n + 1, dtype=np.uint64) * np.uint64(size - 1), cols.reshape(-1).astype(np.uint32))
    gpu_exec.transfer(g)
    for q, kk in ((0, 3), (24, 4)):
        gpu_exec.set_plan(g2.plan_for_preset(q))
        assert gpu_exec.run_gm()["count"] == stride * math.comb(size, kk)
