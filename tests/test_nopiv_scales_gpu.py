"""Unpivoted panels whose pivots' reciprocals are no normal numbers: a matrix scaled by a power of two
has the multipliers of the unscaled one, and so has one whose single pivot is subnormal.

Tolerance: a subnormal reciprocal or pivot keeps 22 of FP32's (51 of FP64's) bits, and an entry takes
at most n updates: 40 n 2^-22 < 1e-3 and 40 n 2^-51 < 1e-11 for n up to 100, of entries of order 1."""

import numpy as np
import pytest

from pyvl_amd import linalg as LA

pytestmark = pytest.mark.gpu


def _factors(n, rng):
    l = np.tril(rng.uniform(-0.4, 0.4, (n, n)) / np.sqrt(n), -1) + np.eye(n)
    u = np.triu(rng.uniform(-0.4, 0.4, (n, n)) / np.sqrt(n), 1) + np.diag(rng.uniform(0.55, 0.9, n))
    return l, u


@pytest.mark.parametrize("prec,top,tol", [("fp32", 127, 1e-3), ("fp64", 1023, 1e-11)])
@pytest.mark.parametrize("n", [1, 17, 64, 100])
def test_large_pivots(prec, top, tol, n):
    """Pivots above 2^(top - 1): 1 / pivot is subnormal."""
    l, u = _factors(n, np.random.default_rng(n))
    a = np.ldexp(l @ u, top)
    assert np.all(np.isfinite(a)) and np.max(np.abs(a)) < 2.0 ** top
    f = LA.LU(n, LA.FP32 if prec == "fp32" else LA.FP64, pivoting=False).factor(a).factors().astype(np.float64)
    assert np.max(np.abs(np.tril(f, -1) - np.tril(l, -1))) <= tol
    assert np.max(np.abs(np.ldexp(np.triu(f), -top) - u)) <= tol


@pytest.mark.parametrize("prec,low,tol", [("fp32", -127, 1e-3), ("fp64", -1023, 1e-11)])
@pytest.mark.parametrize("j", [0, 5, 15])
def test_a_subnormal_pivot(prec, low, tol, j):
    n = 40
    l, u = _factors(n, np.random.default_rng(j))
    s = np.zeros(n, int)
    s[j] = low
    us = np.ldexp(np.ldexp(u, np.minimum(s[:, None], s[None, :])), 0)
    dt = np.float32 if prec == "fp32" else np.float64
    a = (l @ us).astype(dt).astype(np.float64)
    assert abs(dt(us[j, j])) < np.finfo(dt).tiny
    f = LA.LU(n, LA.FP32 if prec == "fp32" else LA.FP64, pivoting=False).factor(a).factors().astype(np.float64)
    assert np.max(np.abs(np.tril(f, -1) - np.tril(l, -1))) <= tol
    assert np.max(np.abs(np.triu(f) - us)) <= tol
    assert np.max(np.abs(np.ldexp(np.triu(f)[: j + 1, j] - us[: j + 1, j], -low))) <= tol
