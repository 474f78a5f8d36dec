"""The closedness check of an upload on both sides of the line between host and
device (2^15 row entries of the sources), at the row lengths where the device's
windows end: a source with a rowless neighbour sends matching down the canonical
path."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LINE = 1 << 15


@pytest.mark.parametrize("d", [1, 2, 63, 64, 65, 255, 256, 257, 2047, 2048, 2049, 5000])
def test_rowless_neighbour_is_found_on_both_sides(g2, gpu_exec, d):
    """a hub and its d neighbours, which know only the hub; the hub as often a
    source as stays within the line, and once more"""
    print("case: upload, both sides, degree", d, flush=True)
    gpu_exec.set_plan(g2.plan_for_preset(0))
    for gone in (None, 0, d - 1):
        deg = np.ones(d + 1, np.uint64)
        deg[0] = d
        cols = np.concatenate((np.arange(1, d + 1), np.zeros(d))).astype(np.uint32)
        if gone is not None:
            deg[1 + gone] = 0
            cols = cols[:-1]
        g = g2.Graph(np.concatenate(([0], np.cumsum(deg))).astype(np.uint64), cols)
        for times in (LINE // d, LINE // d + 1):
            gpu_exec.transfer(g, np.zeros(times, np.uint32))
            r = gpu_exec.run_gm()
            assert r["count"] == 0
            assert r["stats"]["local_bitmap"] == (1 if gone is None or d == 1 else 0), (gone, times)
