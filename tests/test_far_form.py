"""CPU pin of the far form's polynomial (induction_core.hpp, coefficients parsed from the source):
angle / h = (len / B) (1 + s P(s)), s = (len h / B)^2, for points at least four segment lengths
from the midpoint, against 40-digit arithmetic."""

import re
from pathlib import Path

import numpy as np

SRC = (Path(__file__).resolve().parents[1] / "pyvl_amd" / "csrc" / "induction_core.hpp").read_text()


def _coefficients():
    c = {int(k): float(v) for k, v in re.findall(r"kFar(\d) = (-?\d\.\d+e-\d+)", SRC)}
    assert sorted(c) == list(range(1, 8))
    return [c[k] for k in sorted(c)]


def test_far_form_matches_the_angle():
    import mpmath as mp

    mp.mp.dps = 40
    c = _coefficients()
    rng = np.random.default_rng(0)
    worst = 0.0
    for _ in range(4000):
        ln = 10.0 ** rng.uniform(-3, 3)
        # distance of the midpoint in segment lengths, from the rule's edge outwards; any direction
        k = 4.0 * 10.0 ** rng.uniform(0, 3) if rng.random() < 0.7 else 4.0
        th = rng.uniform(0, np.pi)
        t_mid, h = k * ln * np.cos(th), k * ln * np.sin(th)
        t1, t2 = t_mid + ln / 2, t_mid - ln / 2
        b = h * h + t1 * t2
        assert b > 0
        assert (ln * h / b) ** 2 <= 0.0645
        # the exact angle over h at the same (rounded) t1, t2 = t1 - len, h
        T1, H, LN = mp.mpf(t1), mp.mpf(h), mp.mpf(t1) - mp.mpf(t2)
        exact = mp.atan2(LN * H, H * H + T1 * mp.mpf(t2)) / H if h > 0 else LN / (T1 * mp.mpf(t2))
        B = H * H + T1 * mp.mpf(t2)
        S = (LN / B) ** 2 * H * H
        P = mp.mpf(c[6])
        for a in reversed(c[:6]):
            P = P * S + mp.mpf(a)
        worst = max(worst, float(abs(LN / B * (1 + S * P) / exact - 1)))
    # the fit's own bound (4.6e-16) with a margin for the coefficients' rounding
    assert worst < 6e-16
