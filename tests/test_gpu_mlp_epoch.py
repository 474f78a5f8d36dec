"""Mini-batch training at the sizes where the one-workgroup epoch kernel can go wrong: tiles of 16 samples, groups
of 256, a ragged last batch, and both sides of the largest batch it takes."""
import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LR = 2e-3


@pytest.fixture(scope="module")
def dev():
    return importlib.import_module("g2-aimd_amd.device")


def reference(dev, p, batches, epochs):
    """Adam in 64 bits over the gradients of Mlp.grad (its own kernels, pinned against the fp64 network elsewhere)"""
    net = dev.Mlp(seed=1)
    p = p.astype(np.float64)
    m, v, t = np.zeros_like(p), np.zeros_like(p), 0
    for _ in range(epochs):
        sse = 0.0
        for x, y in batches:
            net.set_params(p.astype(np.float32))
            loss, g = net.grad(x, y)
            sse += float(loss) * len(y)
            g = g.astype(np.float64)
            t += 1
            m = 0.9 * m + 0.1 * g
            v = 0.999 * v + 0.001 * g * g
            p -= LR * (m / (1 - 0.9 ** t)) / (np.sqrt(v / (1 - 0.999 ** t)) + 1e-8)
    net.close()
    return p, sse / sum(len(y) for _, y in batches), t


def check(dev, x, y, batch, epochs, batches):
    net = dev.Mlp(seed=9)
    p0 = net.params()
    loss = net.train(x, y, epochs=epochs, batch=batch, lr=LR)
    got = net.params().astype(np.float64)
    net.close()
    ref, ref_loss, steps = reference(dev, p0, batches, epochs)
    err = np.abs(got - ref)
    # An Adam step moves a parameter by about LR whatever the gradient's size, so sums taken in another order
    # (relative 1e-6 or so) show only where a gradient nearly cancels: 99% of the parameters agree to a thousandth
    # of the way moved, and none is further off than the way itself, both sides of it
    assert np.quantile(err, 0.99) <= 1e-3 * LR * steps + 1e-6
    assert err.max() <= 2.5 * LR * steps
    assert abs(loss - ref_loss) <= 1e-3 * abs(ref_loss) + 1e-7


@pytest.mark.parametrize("n", [1, 15, 16, 17, 255, 256, 257, 512, 1000, 1536, 1537])
def test_whole_batches(dev, n):
    """one batch an epoch: the shuffled order only changes the order of sums"""
    print("case: mlp epoch, whole batch", n, flush=True)
    rng = np.random.default_rng(n)
    x = rng.normal(0, 1, (n, 8)).astype(np.float32)
    y = (3 + x @ np.linspace(1, -0.5, 8)).astype(np.float32)
    check(dev, x, y, n, 3, [(x, y)])


@pytest.mark.parametrize("batch,last", [(1, 1), (7, 3), (16, 16), (100, 36), (256, 1), (300, 257), (1536, 17), (1537, 17)])
def test_ragged_epochs(dev, batch, last):
    """equal samples: every order has the same batches, the last one short"""
    print("case: mlp epoch, batches of", batch, "last", last, flush=True)
    n = 3 * batch + last
    x = np.tile(np.random.default_rng(batch).normal(0, 1, 8).astype(np.float32), (n, 1))
    y = np.full(n, 2.5, np.float32)
    b = [(x[:batch], y[:batch])] * 3 + [(x[:last], y[:last])]
    check(dev, x, y, batch, 2, b)
