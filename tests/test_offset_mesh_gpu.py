"""Velocities, matrices and tensors of a mesh far from the origin: only differences of coordinates may
enter, so the error is that of the same mesh at the origin.

Tolerance: the bar of the other parity tests (1e-12 of the largest value).  Both sides start from the
same rounded coordinates; a coordinate of size 1e5 rounds by 1e-11 of the body's radius, ten times
the bar, so a value formed from a rounded absolute position does not pass."""

import numpy as np
import pytest

from oracle import oracle as O
from pyvl_amd import geometry as G
from pyvl_amd.cvl import Mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offset", [0.0, 1e3, 1e5, 1e6])
@pytest.mark.parametrize("n_pts", [1, 129])
def test_velocities_do_not_depend_on_the_origin(offset, n_pts):
    pos, el = G.uv_sphere(32, 16, sigma=1e-2, seed=1)
    rng = np.random.default_rng(n_pts)
    d = rng.normal(size=(n_pts, 3))
    pts = rng.uniform(1.5, 3.0, (n_pts, 1)) * d / np.linalg.norm(d, axis=1, keepdims=True)
    at = offset * np.array([1.0, -0.7, 0.3])
    pos, pts = np.ascontiguousarray(pos + at), np.ascontiguousarray(pts + at)
    m, t = Mesh(pos.shape[0], el), O.mesh_from_elements(pos.shape[0], el)
    circ = rng.normal(size=m.n_surfaces)
    nrm = np.ascontiguousarray(d / np.linalg.norm(d, axis=1, keepdims=True))
    for got, want in ((m.point_velocity(1e-6, pos, circ, pts), O.point_velocity(t, pos, circ, pts, 1e-6)),
                      (m.induction_matrix3(1e-6, pos, pts, nrm), O.induction_matrix3(t, pos, pts, nrm, 1e-6)),
                      (m.induction_matrix(1e-6, pos, pts), O.induction_matrix(t, pos, pts, 1e-6))):
        assert np.max(np.abs(got - want)) <= 1e-12 * np.max(np.abs(want))
