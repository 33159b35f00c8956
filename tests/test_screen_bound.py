"""The screen of the genotype planes' kernels (CPU): its inequality, and the
whole chain in float32 against the information of a pair's 20 evaluations.

KL(p + u || p) <= u^2 / (2 p (1-p)) (1 + k |u|), k = (2 g(s) - 1) / s with s =
min(p, 1-p); so Q = sum over the genotype table's cells of T u^2 (1 + k |u|),
T u = c - p T, is at least 2 p (1-p) m I for every evaluation (a union of
cells).  The constants are screen_consts's, restated here.
"""
import math

import numpy as np
import pytest

from test_filter_bounds import mi_nats
from test_filter_slope import g


def consts(n0, n1):
    n = n0 + n1
    p = n0 / n
    s = min(p, 1.0 - p)
    k = (2.0 * g(s) - 1.0) / s * (1.0 + 1e-6)
    bits = 0
    while bits < 16 and n >= 1 << bits:
        bits += 1
    start = 2.0 ** -min(24 - bits, 12)
    q = 2.0 * p * (1.0 - p) * (1.0 - 1e-4)
    return [np.float32(v) for v in (p, k, q * n, start, 18.0 * start * (1.0 + 2.0 * k) + 1e-3)]


def kl(a, p):
    return sum(x * math.log(x / y) if x > 0.0 else 0.0 for x, y in ((a, p), (1.0 - a, 1.0 - p)))


def test_cell_bound():
    for p in [1e-4, 1e-3, 0.01, 0.03, 0.1, 0.2, 0.3, 0.45, 0.5, 0.6, 0.8, 0.97, 0.9999]:
        s = min(p, 1.0 - p)
        k = (2.0 * g(s) - 1.0) / s
        for a in np.concatenate([np.linspace(0.0, 1.0, 4001), p + s * np.linspace(-1e-3, 1e-3, 201)]):
            u = float(a) - p
            b = u * u / (2.0 * p * (1.0 - p)) * (1.0 + k * abs(u))
            assert kl(float(a), p) <= b * (1.0 + 1e-9) + 1e-15, (p, a)


@pytest.mark.parametrize("n", [2, 15, 16, 4095, 4096, 8192, 32767, 32768, 46340])
def test_start_is_exact(n):
    """A count of up to n and three times the start are whole multiples of it
    below 2^24 of it."""
    start = float(consts(n - n // 3, n // 3)[3]) if n >= 3 else float(consts(1, 1)[3])
    for c in (0, 1, n // 2, n - 1, n):
        assert float(np.float32(c + start)) == c + start
    assert (n + start) / start <= 2 ** 24


@pytest.mark.parametrize("n0,n1", [(20, 20), (60, 5), (130, 126), (1229, 819), (1900, 148), (5734, 2458),
                                   (23170, 23170), (44000, 2340)])
def test_no_evaluation_is_screened_out(n0, n1):
    """Right side for the best evaluation's own information: the pair passes."""
    f = np.float32
    p, k, qm, start, sub = consts(n0, n1)
    rng = np.random.default_rng(n0 + 7 * n1)
    n = n0 + n1
    carries = [np.array([1, 1, 0], bool), np.array([0, 1, 1], bool)]
    for rep in range(400):
        fa, fb = rng.uniform(0.01, 0.99, 2)
        ga, gb = (np.array([(1 - x) ** 2, 2 * x * (1 - x), x * x]) for x in (fa, fb))
        miss = rng.choice([0.0, 0.02, 0.2])
        pr = np.zeros((4, 4))
        pr[:3, :3] = np.outer(ga, gb)
        effect = np.ones((4, 4)) * 0.25
        effect[:3, :3] = rng.dirichlet(np.full(9, rng.choice([0.1, 1.0, 20.0]))).reshape(3, 3)
        tab = []
        for c, size in ((0, n0), (1, n1)):
            w = pr * (effect if c == 1 and rep % 2 else 1.0)
            w = w / w.sum() * (1.0 - miss) ** 2
            w[3, :3] = miss * (1.0 - miss) * w[:3, :3].sum(0) / max(w[:3, :3].sum(), 1e-30)
            w[:3, 3] = miss * (1.0 - miss) * w[:3, :3].sum(1) / max(w[:3, :3].sum(), 1e-30)
            w[3, 3] = 0.0
            w[3, 3] = max(0.0, 1.0 - w.sum())
            tab.append(rng.multinomial(size, (w / w.sum()).ravel()).reshape(4, 4))
        c0, c1 = tab[0][:3, :3], tab[1][:3, :3]
        y, z = int(c0.sum()), int(c1.sum())
        if y + z == 0:
            continue
        best = 0.0
        for a in carries:
            for b in carries:
                A, B = a[:, None] & np.ones(3, bool), b[None, :] & np.ones((3, 1), bool)
                for ev in (A & B, ~A & B, A & ~B, ~(A | B), A ^ B):
                    best = max(best, mi_nats(int(c0[ev].sum()), int(c1[ev].sum()), y, z))
        # the kernel's right side: R (1 - both variants' missing shares) - sub
        R = f(best) * qm
        ma = f((tab[0][3].sum() + tab[1][3].sum()) / n)
        mb = f((tab[0][:, 3].sum() + tab[1][:, 3].sum()) / n)
        rhs = f(f(f(R - sub) - R * mb) - R * ma)
        q = f(0.0)
        for T, c in zip((c0 + c1).ravel(), c0.ravel()):
            T, c = f(T) + start, f(c)
            e = f(c - p * T)
            u = f(e / T)
            q = f(q + f(e * u) * f(f(1.0) + k * abs(u)))
        assert q > rhs, (n0, n1, rep, float(q), float(rhs))
