"""Inference whose output buffer is, or overlaps, the input buffer: the outputs are those of separate
buffers, bit for bit (both paths form the same products in the same order)."""

import ctypes as C

import numpy as np
import pytest

from pyvl_amd import DeviceArray, _lib
from pyvl_amd import learned as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d_in,batch,at", [(18, 33, 0), (18, 20000, 0), (18, 5000, 7), (1, 700, 0), (1, 700, 64)])
def test_forward_over_its_inputs(d_in, batch, at):
    """The output starts `at` floats into the input (d_in 1 and 64: past its first rows)."""
    net = L.MLP(d_in, 64, 3, seed=2)
    x = np.random.default_rng(batch).normal(size=(batch, d_in)).astype(np.float32)
    want = net.forward(DeviceArray.from_numpy(x)).numpy()
    buf = np.zeros(batch * d_in + at, np.float32)
    buf[:batch * d_in] = x.ravel()
    d = DeviceArray.from_numpy(buf)
    p = C.cast(d.cptr, C.c_void_p).value
    _lib.call("pvl_mlp_forward", net._h, C.c_void_p(p), C.c_void_p(p + 4 * at), C.c_int(batch))
    assert np.array_equal(d.numpy()[at:at + batch], want)
