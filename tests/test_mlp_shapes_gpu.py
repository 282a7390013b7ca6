"""The network's fused pass and sliced weight gradients against the oracle at the shapes where they
can go wrong: input counts that are no multiple of 8, wider inputs than layers, widths that are no
multiple of 16 or 32, two to five layers, batches below a workgroup's 32 samples, odd ones, and
enough for several slices; width 300 and five layers of 256 take the general kernels.

Tolerances are those of the other network tests (BF16 operands, FP32 accumulation): 1e-2 for the
output, 2e-2 per layer for the gradients, against the oracle that rounds at the same points."""

import numpy as np
import pytest

from oracle import mlp_oracle as MO
from pyvl_amd import DeviceArray
from pyvl_amd import learned as L

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(b))


@pytest.mark.parametrize("d_in,width,layers,batch", [(18, 256, 4, 1), (18, 256, 4, 33), (18, 256, 4, 1300),
                                                     (5, 64, 3, 100), (40, 24, 3, 31), (16, 40, 2, 65),
                                                     (7, 50, 4, 257), (18, 256, 5, 70), (18, 300, 3, 64)])
def test_forward_and_gradient_match_oracle(d_in, width, layers, batch):
    dims = (d_in,) + (width,) * (layers - 1) + (1,)
    net = L.MLP(d_in, width, layers, seed=3)
    rng = np.random.default_rng(batch + width)
    p = net.get_params().astype(np.float64)
    for _, b in net.unpack(p):
        b[:] = rng.normal(0.0, 0.1, b.size)
    net.set_params(p.astype(np.float32))
    p = net.get_params().astype(np.float64)
    x = rng.normal(size=(batch, d_in)).astype(np.float32)
    t = (np.sin(x[:, 0]) + x[:, 1] * x[:, 2]).astype(np.float32)
    dx, dt = DeviceArray.from_numpy(x), DeviceArray.from_numpy(t)
    y_ref, _, _ = MO.forward(p, dims, x, bf16=True)
    assert _rel(net.forward(dx).numpy(), y_ref) < 1e-2
    g, loss = net.gradient(dx, dt)
    loss_ref, g_ref = MO.loss_and_gradient(p, dims, x, t, bf16=True)
    assert abs(loss - loss_ref) <= 1e-2 * loss_ref
    off = 0
    for n_in, n_out in zip(dims[:-1], dims[1:]):
        for sl in (slice(off, off + n_in * n_out), slice(off + n_in * n_out, off + n_in * n_out + n_out)):
            assert _rel(g[sl], g_ref[sl]) < 2e-2, sl
        off += n_in * n_out + n_out
    # weights changed by a step: the backward pass uses the new ones
    net.train_step(dx, dt, 1e-2)
    p1 = net.get_params().astype(np.float64)
    g1, _ = net.gradient(dx, dt)
    _, g1_ref = MO.loss_and_gradient(p1, dims, x, t, bf16=True)
    assert _rel(g1, g1_ref) < 2e-2
