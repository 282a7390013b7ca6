"""Pivoted panels shared by several workgroups: interchanges inside a sub-block of eight columns, out
of it, and chained through it, at the sizes where the panel width, the groups and the last sub-block
change, against LAPACK (pivots equal, factors to the rounding of the updates)."""

import numpy as np
import pytest
import scipy.linalg as sla

from pyvl_amd import linalg as LA

pytestmark = pytest.mark.gpu


def _matrix(kind, n, rng):
    u = np.triu(rng.normal(size=(n, n)) / np.sqrt(n), 1) + np.diag(2.0 + rng.uniform(size=n))
    if kind == "reverse":
        return u[::-1]
    if kind == "shift":  # every column displaces the row that the one before it displaced
        return np.roll(u, 1, axis=0)
    if kind == "blocks":  # permuted inside every eight rows
        p = np.arange(n)
        for k in range(0, n, 8):
            p[k:k + 8] = k + rng.permutation(min(8, n - k))
        return u[p]
    if kind == "ties":
        return rng.integers(-2, 3, size=(n, n)).astype(float) + 4.0 * np.eye(n)[rng.permutation(n)]
    return rng.normal(size=(n, n))


@pytest.mark.parametrize("n", [1025, 1063, 2049, 2117])
@pytest.mark.parametrize("kind", ["reverse", "shift", "blocks", "normal", "ties"])
def test_grouped_panel_interchanges(kind, n):
    a = np.ascontiguousarray(_matrix(kind, n, np.random.default_rng(n)))
    lu_ref, piv_ref = sla.lu_factor(a)
    h = LA.LU(n).factor(a)
    if kind == "ties":  # rounding may break a tie either way after the first column
        assert h.pivots()[0] == piv_ref[0]
        b = np.ones(n)
        x = h.solve(b)
        assert np.linalg.norm(a @ x - b) <= 1e-9 * np.linalg.norm(a) * np.linalg.norm(x)
        return
    assert np.array_equal(h.pivots(), piv_ref)
    assert np.linalg.norm(h.factors() - lu_ref) <= 1e-12 * np.linalg.norm(lu_ref)


@pytest.mark.parametrize("kind", ["reverse", "shift", "blocks"])
def test_grouped_panel_interchanges_fp32(kind):
    n = 2117
    a = np.ascontiguousarray(_matrix(kind, n, np.random.default_rng(n)))
    lu_ref, piv_ref = sla.lu_factor(a.astype(np.float32))
    h = LA.LU(n, LA.FP32).factor(a)
    assert np.array_equal(h.pivots(), piv_ref)
    assert np.linalg.norm(h.factors() - lu_ref) <= 1e-5 * np.linalg.norm(lu_ref)


def test_grouped_panel_zero_column():
    n = 1100
    a = np.random.default_rng(1).normal(size=(n, n))
    a[:, 13] = 0.0
    with pytest.warns(RuntimeWarning):
        assert LA.LU(n).factor(a).info == 14
