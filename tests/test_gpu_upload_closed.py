"""What an upload finds out about its view on the device, at the sizes where the kernels' row windows end: a source
with a rowless neighbour (first, last, none) sends matching down the canonical path, whatever the row's length."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [1, 2, 63, 64, 65, 255, 256, 257, 2047, 2048, 2049, 5000])
def test_rowless_neighbour_is_found(g2, gpu_exec, d):
    """a hub and its d neighbours, which know only the hub; a triangle's root has degree >= 2"""
    print("case: upload, rowless neighbour, degree", d, flush=True)
    for gone in (None, 0, d - 1):
        deg = np.ones(d + 1, np.uint64)
        deg[0] = d
        cols = np.concatenate((np.arange(1, d + 1), np.zeros(d))).astype(np.uint32)
        if gone is not None:
            deg[1 + gone] = 0
            cols = cols[:-1]
        rp = np.concatenate(([0], np.cumsum(deg))).astype(np.uint64)
        for sources in ([0], [d, 0, 1]):
            gpu_exec.transfer(g2.Graph(rp, cols), np.array(sources, np.uint32))
            gpu_exec.set_plan(g2.plan_for_preset(0))
            r = gpu_exec.run_gm()
            assert r["count"] == 0
            assert r["stats"]["local_bitmap"] == (1 if gone is None or d == 1 else 0)


def test_ids_out_of_range_are_refused_anywhere(g2, gpu_exec):
    """one bad id among many, at the ends and in the tail of the vectorised check"""
    print("case: upload, id out of range", flush=True)
    n = 1000
    rp = np.arange(0, 37 * (n + 1), 37, dtype=np.uint64)
    cols = (np.arange(37 * n) % n).astype(np.uint32)
    for at in (0, 1, 17, 20000, 37 * n - 2, 37 * n - 1):
        for bad in (n, 0x80000000, 0xFFFFFFFF):
            c = cols.copy()
            c[at] = bad
            with pytest.raises(RuntimeError, match="column id"):
                gpu_exec.transfer(g2.Graph(rp, c))
    for at in (0, n // 2, n - 1):
        s = np.arange(n, dtype=np.uint32)
        s[at] = n
        with pytest.raises(RuntimeError, match="source id"):
            gpu_exec.transfer(g2.Graph(rp, cols), s)
