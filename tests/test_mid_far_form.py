"""CPU pins of the far form that the FP64 assembly and the point-velocity sums take from two segment
lengths off the midpoint (mid_far and mid_holds in induction_core.hpp, parsed from the source): both copies
of the polynomial, its error against 40-digit arithmetic over the whole range that the test lets through,
and the test's bit pattern."""

import re
import struct
from pathlib import Path

import numpy as np

SRC = (Path(__file__).resolve().parents[1] / "pyvl_amd" / "csrc" / "induction_core.hpp").read_text()
NUM = r"-?\d\.\d+e-\d+"


def _copies():
    body = SRC[SRC.index("double mid_far("):]
    body = body[:body.index("\n}\n")]
    first = float(re.search(rf"double p = ({NUM})", body).group(1))
    steps = [float(x) for x in re.findall(rf"fma_step<true>\(p, u, ({NUM})\)", body)]
    regs = [float(x) for x in re.findall(rf'"s"\(({NUM})\)', body)]
    return first, steps, regs, body


def test_both_copies_hold_the_same_coefficients_in_order():
    first, steps, regs, body = _copies()
    assert len(steps) == 10 and steps == regs
    used = re.findall(r"v_fma_f64 %0, %0, %1, %(\d+)", body)
    assert [int(k) for k in used] == list(range(2, 12))


def test_mid_far_matches_the_angle():
    import mpmath as mp

    mp.mp.dps = 40
    first, steps, _, _ = _copies()
    rng = np.random.default_rng(0)
    worst = 0.0
    for i in range(4000):
        ln = 10.0 ** rng.uniform(-3, 3)
        k = 2.0 if i % 3 == 0 else 2.0 * 10.0 ** rng.uniform(0, 3)  # midpoint distance in segment lengths
        th = rng.uniform(0, np.pi)
        t_mid, h = mp.mpf(k * ln * np.cos(th)), mp.mpf(k * ln * np.sin(th))
        L = mp.mpf(ln)
        b = h * h + (t_mid + L / 2) * (t_mid - L / 2)
        assert L * L / b <= mp.mpf("0.26667")
        q = L / b
        u = h * h * q * q
        assert u <= mp.mpf("0.2845")
        p = mp.mpf(first)
        for c in steps:
            p = p * u + mp.mpf(c)
        exact = mp.atan2(L * h, b) / h
        worst = max(worst, float(abs(q * (1 + u * p) / exact - 1)))
    # the fit's own bound (3.2e-16) with a margin for the coefficients' rounding
    assert worst < 5e-16


def test_mid_holds_lets_through_two_lengths_and_nothing_else():
    word = int(re.search(r"< (0x[0-9A-Fa-f]+)u;", SRC[SRC.index("bool mid_holds("):]).group(1), 16)

    def holds(x):
        return (struct.unpack("<Q", struct.pack("<d", x))[0] >> 32) < word

    assert word == struct.unpack("<Q", struct.pack("<d", 1.0 / 3.75))[0] >> 32
    assert holds(0.0) and holds(5e-324) and holds(0.2666)
    for x in (1.0 / 3.75, 0.27, 1.0, np.inf, np.nan, -0.0, -1e-300, -1.0, -np.inf):
        assert not holds(x)


def test_mid_reach_takes_lengths_whose_squares_are_normal_numbers():
    body = SRC[SRC.index("double mid_reach("):]
    lo, hi, lo2 = (int(x, 16) for x in re.findall(r"(0x[0-9A-F]+)u", body[:body.index(";", body.index("in_range"))]))
    assert lo == lo2

    def in_range(x):
        return ((struct.unpack("<Q", struct.pack("<d", x))[0] >> 32) - lo) % 2**32 < hi - lo

    for x in (1e-99, 1e-6, 1.0, 1e99, 2.0**-332, 2.0**332.999):
        assert in_range(x) and np.finfo(float).tiny < 3.75 * (x * x) < np.inf
    for x in (0.0, 5e-324, 1e-101, 2.0**333, 1e300, np.inf, np.nan):
        assert not in_range(x)
