"""Triangular solves of rows so unlike in scale that u_ik / u_kk leaves the range of the type: powers
of two on the rows of a system leave its solution as it is."""

import numpy as np
import pytest
import scipy.linalg as sla

from pyvl_amd import linalg as LA

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,n", [("fp64", 2), ("fp64", 65), ("fp64", 200), ("fp32", 64), ("fp32", 131)])
def test_rows_of_unlike_scales(prec, n):
    """Upper triangular (its own factor), well conditioned; rows scaled up and down in turn.  The
    substitution's error is a few n eps of x: 1e-12 in FP64, 1e-5 in FP32."""
    rng = np.random.default_rng(n)
    dt, e = (np.float64, 600) if prec == "fp64" else (np.float32, 70)
    u = (np.triu(rng.normal(size=(n, n)) / np.sqrt(n), 1) + np.diag(2.0 + rng.uniform(size=n))).astype(dt)
    b = rng.normal(size=n).astype(dt)
    x_ref = sla.solve_triangular(u.astype(np.float64), b.astype(np.float64))
    for first in (e, -e):
        s = np.where(np.arange(n) % 2 == 0, 2.0 ** first, 2.0 ** -first)
        h = LA.LU(n, LA.FP64 if prec == "fp64" else LA.FP32).factor(u.astype(np.float64) * s[:, None])
        x = h.solve((b * s).astype(dt)).astype(np.float64)
        assert np.max(np.abs(x - x_ref)) < (1e-12 if prec == "fp64" else 1e-5) * np.max(np.abs(x_ref))
