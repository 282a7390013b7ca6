"""Error of single-right-hand-side solves, with triangular systems (their own factors) against extended
precision.  A row's terms are summed apart and subtracted once, so an entry takes the rounding of one
difference and one quotient, 0.29 units in the last place each in the mean square, passed on by a
factor below 1.5 (rows of off-diagonal norm below 0.5 of the diagonal), and the smaller ones of its sum:
below one unit in the mean square.  Subtracted term by term from the running value, the 64 roundings of a block
add up to more."""

import numpy as np
import pytest

from pyvl_amd import linalg as LA

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("n", [64, 65, 300])
@pytest.mark.parametrize("lower", [False, True])
def test_rounding_of_a_solve(prec, n, lower):
    dt = np.float64 if prec == "fp64" else np.float32
    err = []
    for seed in range(16):
        rng = np.random.default_rng([n, seed])
        g = np.triu(rng.normal(size=(n, n)) / np.sqrt(n), 1)
        # lower: unit diagonal with small multipliers (nothing interchanged), U the identity
        a = (0.4 * g.T + np.eye(n) if lower else g + np.diag(2.0 + rng.uniform(size=n))).astype(dt)
        b = rng.normal(size=n).astype(dt)
        x = LA.LU(n, LA.FP64 if prec == "fp64" else LA.FP32, pivoting=False).factor(a.astype(float)).solve(b)
        al, want = a.astype(np.longdouble), np.zeros(n, np.longdouble)
        for i in range(n) if lower else range(n - 1, -1, -1):
            want[i] = (b[i] - al[i] @ want) / al[i, i]
        err.append(np.linalg.norm((x - want).astype(float)) / np.linalg.norm(want.astype(float)))
    assert np.sqrt(np.mean(np.square(err))) <= 1.0 * np.finfo(dt).eps


@pytest.mark.parametrize("prec,e", [("fp64", 1000), ("fp32", 110)])
@pytest.mark.parametrize("n", [1, 64, 131])
def test_diagonals_out_of_the_corrections_range(prec, e, n):
    """Rows scaled by powers of two beyond 2^900 (FP32 2^90) either way divide at every step; the solution is
    that of the unscaled system bit for bit, as every operation scales."""
    dt = np.float64 if prec == "fp64" else np.float32
    rng = np.random.default_rng(n)
    u = (np.triu(rng.normal(size=(n, n)) / np.sqrt(n), 1) + np.diag(2.0 + rng.uniform(size=n))).astype(dt)
    b = rng.uniform(0.5, 2.0, n).astype(dt)
    s = np.where(np.arange(n) % 3 == 0, 2.0 ** e, np.where(np.arange(n) % 3 == 1, 2.0 ** -e, 1.0))
    p = LA.FP64 if prec == "fp64" else LA.FP32
    want = LA.LU(n, p, pivoting=False).factor(u.astype(float)).solve(b)
    got = LA.LU(n, p, pivoting=False).factor(u.astype(float) * s[:, None]).solve((b * s).astype(dt))
    assert np.array_equal(got, want)
