"""Training: the epoch in one launch (batches of up to 1536 samples) against the
three launches of a step that larger batches take.  The products and the order of
the sums are the same, so parameters and losses are equal bit for bit: no
tolerance.  A batch larger than the samples there are is one step of all of them
on the three-launch path, whatever their number."""
import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

THREE_LAUNCHES = 2000  # a batch size beyond the one-launch path's


@pytest.fixture(scope="module")
def dev():
    return importlib.import_module("g2-aimd_amd.device")


def pair(dev, seed):
    """two models with the same parameters"""
    a, b = dev.Mlp(device=0, seed=seed), dev.Mlp(device=0, seed=seed)
    assert np.array_equal(a.params(), b.params())
    return a, b


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 255, 256, 257, 511, 513, 1000, 1535, 1536])
def test_one_step_an_epoch(dev, n):
    """random samples, five epochs of one step"""
    print("case: training paths, one step of", n, flush=True)
    rng = np.random.default_rng(n)
    x = rng.standard_normal((n, 8)).astype(np.float32)
    y = (x @ np.linspace(1, -0.5, 8) + np.maximum(x[:, 0] * x[:, 3], 0)).astype(np.float32)
    one, three = pair(dev, 3)
    for epochs in (1, 4):
        assert one.train(x, y, epochs=epochs, batch=n, lr=2e-3) == three.train(x, y, epochs=epochs, batch=THREE_LAUNCHES, lr=2e-3)
        assert np.array_equal(one.params(), three.params())


@pytest.mark.parametrize("n,batch", [(5, 1), (50, 16), (513, 256), (1000, 300), (1025, 512), (3000, 1536), (3073, 1536)])
def test_many_steps_an_epoch(dev, n, batch):
    """equal samples, so that a step does not depend on the epoch's order: the
    steps one by one, the last one ragged"""
    print("case: training paths,", n, "samples in batches of", batch, flush=True)
    rng = np.random.default_rng(n)
    x = np.tile(rng.standard_normal((1, 8)).astype(np.float32), (n, 1))
    y = np.full(n, 1.7, np.float32)
    one, three = pair(dev, 5)
    for _ in range(2):
        one.train(x, y, epochs=1, batch=batch, lr=2e-3)
        for b in range(0, n, batch):
            m = min(batch, n - b)
            three.train(x[:m], y[:m], epochs=1, batch=THREE_LAUNCHES, lr=2e-3)
        assert np.array_equal(one.params(), three.params())
