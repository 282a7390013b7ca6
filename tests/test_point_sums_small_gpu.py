"""FP64 point sums on both sides of the size where a lane takes two points (32 chunks of lines: 32 blocks of
128), a single point, and blocks that are not full, near and far points mixed, against the oracle: the
bar of the other parity tests (1e-12 of the largest velocity)."""

import numpy as np
import pytest

from oracle import oracle as O
from pyvl_amd import geometry as G
from pyvl_amd.cvl import Mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_pts", [1, 63, 65, 129, 3968, 3969])
def test_one_and_two_points_per_lane(n_pts):
    pos, el = G.uv_sphere(64, 64, sigma=1e-3, seed=3)
    m, t = Mesh(pos.shape[0], el), O.mesh_from_elements(pos.shape[0], el)
    assert (m.n_lines + 255) // 256 == 32
    rng = np.random.default_rng(n_pts)
    d = rng.normal(size=(n_pts, 3))
    r = np.where(np.arange(n_pts) % 2 == 0, 1.02, rng.uniform(1.1, 4.0, n_pts))[:, None]
    pts = np.ascontiguousarray(r * d / np.linalg.norm(d, axis=1, keepdims=True))
    circ = rng.normal(size=m.n_surfaces)
    want = O.point_velocity(t, pos, circ, pts, 1e-6)
    assert np.max(np.abs(m.point_velocity(1e-6, pos, circ, pts) - want)) <= 1e-12 * np.max(np.abs(want))
