"""Memory of a training batch: the fused pass needs the hidden layers' inputs and every layer's output
error in BF16 (2 bytes each per sample and unit) and no pre-activations.  The general kernels' buffers
come when a call needs them, in any order of batch sizes."""

import numpy as np
import pytest
import torch

from pyvl_amd import DeviceArray
from pyvl_amd import learned as L

pytestmark = pytest.mark.gpu


def test_fused_training_holds_no_pre_activations():
    batch, d_in, width, layers = 1 << 17, 18, 256, 4
    net = L.MLP(d_in, width, layers, seed=1)
    rng = np.random.default_rng(0)
    x = DeviceArray.from_numpy(rng.normal(size=(batch, d_in)).astype(np.float32))
    t = DeviceArray.from_numpy(rng.normal(size=batch).astype(np.float32))
    net.gradient(DeviceArray.from_numpy(np.zeros((64, d_in), np.float32)),
                 DeviceArray.from_numpy(np.zeros(64, np.float32)))
    before = torch.cuda.mem_get_info()[0]
    net.gradient(x, t)
    used = before - torch.cuda.mem_get_info()[0]
    needed = 2 * 2 * (layers - 1) * width * batch + 2 * batch
    assert used <= needed + (64 << 20), (used, needed)


@pytest.mark.parametrize("width", [64, 300])
def test_batches_in_any_order(width):
    """Inference, gradients and inference over the inputs' own buffer at growing and shrinking batches."""
    net = L.MLP(18, width, 3, seed=4)
    rng = np.random.default_rng(width)
    x = rng.normal(size=(3000, 18)).astype(np.float32)
    t = DeviceArray.from_numpy(rng.normal(size=3000).astype(np.float32))
    want = net.forward(DeviceArray.from_numpy(x)).numpy()
    first = {}
    for n in (33, 3000, 700, 1500, 33, 3000, 700):
        d = DeviceArray.from_numpy(np.ascontiguousarray(x[:n]))
        g, loss = net.gradient(d, DeviceArray.from_numpy(t.numpy()[:n]))
        g0, loss0 = first.setdefault(n, (g.copy(), loss))
        assert np.allclose(g, g0, rtol=1e-5, atol=1e-6) and abs(loss - loss0) <= 1e-5 * loss0
        net.forward(d, d)
        assert np.array_equal(d.numpy().ravel()[:n], want[:n])
