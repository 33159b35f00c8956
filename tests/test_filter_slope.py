"""The filters' class-fraction coefficient (CPU, exact math).

I <= g(p) chi2/m with p = min(y, z)/m, g(p) = -ln(1-p) (1-p)/p, and the
tangent h0 + h1 min(y, z) <= 1/g(p) that the kernels use for tables of a
scan with classes of n0 >= y and n1 >= z samples (chi2_slope, restated here
with its float32 results).
"""
import math

import numpy as np
import pytest

from test_filter_bounds import H, all_small_tables, chi2_over_m, lchoose, mi_nats, tables


def g(p):
    return 1.0 - p / 2 if p < 1e-9 else -math.log1p(-p) * (1.0 - p) / p


def slope(n0, n1):
    n = n0 + n1
    p = min(n0, n1) / n if n else 0.0
    h, d = 1.0, 0.5
    if p > 0.0:
        h = 1.0 / g(p)
        d = 0.5 if p < 1e-4 else (-math.log1p(-p) / (p * p) - 1.0 / p) / (g(p) * g(p))
    return np.float32(h - d * p - 1e-6), np.float32(d / n * (1.0 - 1e-6)) if n else np.float32(0.0)


def test_information_below_class_fraction_bound():
    rng = np.random.default_rng(11)
    for w, x, y, z in list(all_small_tables(14)) + list(tables(rng, 20000, 5000)):
        b = g(min(y, z) / (y + z)) * chi2_over_m(w, x, y, z)
        assert mi_nats(w, x, y, z) <= b + 1e-12 * max(1.0, b), (w, x, y, z)


@pytest.mark.parametrize("n0,n1", [(0, 0), (0, 7), (1, 1), (1, 46339), (45, 44), (128, 128),
                                   (465, 273), (1024, 1024), (5734, 2458), (2, 20000),
                                   (23170, 23170), (6000, 14001)])
def test_tangent_below_inverse(n0, n1):
    h0, h1 = slope(n0, n1)
    ys = np.unique(np.linspace(0, n0, 200).astype(int))
    zs = np.unique(np.linspace(0, n1, 200).astype(int))
    for y in ys:
        for z in zs:
            if y + z == 0:
                continue
            k = np.float32(h0 + np.float32(h1 * np.float32(min(y, z))))
            assert float(k) <= 1.0 / g(min(y, z) / (y + z)), (n0, n1, y, z)


def ln_p_obs(w, x, y, z):
    return lchoose(y, w) + lchoose(z, x) - lchoose(y + z, w + x)


def test_fisher_probability_above_bound():
    """ln P(obs) >= -m I - ln(2.55 m) / 2, and its binomial lower bound."""
    rng = np.random.default_rng(12)
    for w, x, y, z in list(all_small_tables(14)) + list(tables(rng, 20000, 5000)):
        m = y + z
        lp = ln_p_obs(w, x, y, z)
        assert lp >= -m * mi_nats(w, x, y, z) - 0.5 * math.log(2.55 * m) - 1e-9 * max(1.0, -lp), (w, x, y, z)
    for n in list(range(2, 200)) + [1000, 4097, 46340]:
        for k in range(1, n) if n < 200 else np.linspace(1, n - 1, 97).astype(int):
            k = int(k)
            lb = n * H(k / n) + 0.5 * math.log(n / (8.0 * k * (n - k)))
            assert lchoose(n, k) >= lb - 1e-9 * max(1.0, lb), (n, k)


def test_float_information_within_margin():
    """entropy_admits: float32 sums of t log2 t within 8e-6 m log2 m (+ 1e-6)
    of the exact -I m."""
    f = np.float32
    rng = np.random.default_rng(13)

    def t(v):
        return f(0) if v == 0 else f(f(v) * np.log2(f(v)))

    for w, x, y, z in list(all_small_tables(9)) + list(tables(rng, 20000, 20000)):
        m = y + z
        s = f(f(f(t(y) + t(z)) - t(m)) + f(t(w + x) + t(m - w - x))) - \
            f(f(t(w) + t(y - w)) + f(t(x) + t(z - x)))
        exact = -m * mi_nats(w, x, y, z) / math.log(2.0)
        assert abs(float(s) - exact) <= 8e-6 * m * math.log2(max(m, 1)) + 1e-6, (w, x, y, z)
