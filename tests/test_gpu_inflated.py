"""Scans whose evaluations are far from a chance ranking: a threshold guessed
for unrelated phenotypes admits nearly all of them (phenotypes that follow two
ancestries) or too few (variants mostly monomorphic).  The guessed band stops
when its list is full and is redone in a few pieces under a threshold of its
own records, or the scan is run without the guess; single scans, the
allocation-free scan and the batch engine.  Against the oracle, or the
band-by-band loop without a guess; the number of bands is bounded."""
import numpy as np
import pytest

import gepicount_amd as ge
from oracle import oracle as orc
from test_gpu_bands import band_by_band
from test_gpu_parity import assert_same

pytestmark = pytest.mark.gpu


def ancestry_panel(seed, n_var, n, miss=0.01):
    """Two populations with their own allele frequencies; nine cases in ten are of one."""
    rng = np.random.default_rng(seed)
    pop = rng.random(n) < 0.5
    base, d = rng.uniform(0.1, 0.5, n_var), rng.normal(0, 0.15, n_var)
    f = np.where(pop[None, :], np.clip(base + d, 0.02, 0.98)[:, None], np.clip(base - d, 0.02, 0.98)[:, None])
    g = (rng.random((n_var, n)) < f).astype(np.uint8) + (rng.random((n_var, n)) < f)
    codes = np.array([3, 2, 0], np.uint8)[g]
    codes[rng.random((n_var, n)) < miss] = 1
    m0, m1 = orc.masks_from_classes((rng.random(n) < np.where(pop, 0.9, 0.1)).astype(int))
    return (*orc.planes_from_codes(codes), m0, m1)


def monomorphic_panel(seed, n_var, n, step):
    """All but every step-th variant monomorphic."""
    rng = np.random.default_rng(seed)
    codes = np.zeros((n_var, n), np.uint8)
    codes[::step] = rng.choice(np.array([0, 2, 3], np.uint8), size=codes[::step].shape)
    m0, m1 = orc.masks_from_classes(rng.integers(0, 2, n))
    return (*orc.planes_from_codes(codes), m0, m1)


@pytest.mark.parametrize("ffun", [0, 1])
@pytest.mark.parametrize("n_var,n,k", [(2500, 400, 100), (2500, 400, 3000), (5200, 150, 1000)])
@pytest.mark.parametrize("noalloc", [False, True])
def test_ancestry(monkeypatch, n_var, n, k, ffun, noalloc):
    """A whole scan in the guessed band, and a pilot before larger bands."""
    print("case inflated", n_var, n, k, ffun, noalloc, flush=True)
    bits, valid, m0, m1 = ancestry_panel(41, n_var, n)
    with ge.Panel.from_planes(bits, valid, n) as panel:
        got, st = (panel.scan_noalloc if noalloc else panel.scan)(m0, m1, topmost=k, ffun=ffun)
        ref, _ = band_by_band(monkeypatch, panel, m0, m1, k, ffun, 64)
    assert_same(got, ref, "ancestry")
    # (the allocation-free scan's short lists do not hold every guess)
    assert noalloc or st["pend_overflows"] + st["cand_overflows"] > 0
    assert st["bands"] <= 24, st


@pytest.mark.parametrize("ffun", [0, 1])
@pytest.mark.parametrize("k", [200, 10000])
def test_monomorphic(monkeypatch, k, ffun):
    print("case monomorphic", k, ffun, flush=True)
    bits, valid, m0, m1 = monomorphic_panel(43, 1500, 130, 90)
    with ge.Panel.from_planes(bits, valid, 130) as panel:
        got, st = panel.scan(m0, m1, topmost=k, ffun=ffun)
        ref, _ = band_by_band(monkeypatch, panel, m0, m1, k, ffun, 64)
    assert_same(got, ref, "monomorphic")
    assert st["bands"] <= 12, st


@pytest.mark.parametrize("ffun", [0, 1])
def test_rare(monkeypatch, ffun):
    """Alleles of at most 1%, whose scores are few and far apart: the guess finds
    a part of the ranking (a looser one follows) or next to nothing of it."""
    print("case rare", ffun, flush=True)
    rng = np.random.default_rng(5)
    f = rng.uniform(0.002, 0.01, 1024)[:, None]
    g = (rng.random((1024, 256)) < f).astype(np.uint8) + (rng.random((1024, 256)) < f)
    bits, valid = orc.planes_from_codes(np.array([3, 2, 0], np.uint8)[g])
    m0, m1 = orc.masks_from_classes((rng.random(256) < 0.4).astype(int))
    with ge.Panel.from_planes(bits, valid, 256) as panel:
        got, st = panel.scan(m0, m1, topmost=100, ffun=ffun)
        ref, _ = band_by_band(monkeypatch, panel, m0, m1, 100, ffun, 64)
    assert_same(got, ref, "rare")
    assert st["bands"] <= 6, st


def test_batch():
    """Guesses that overflow and that fail next to ones that hold, both
    objectives, on allele and genotype planes, in one batch."""
    print("case inflated batch", flush=True)
    made = []
    for i in range(8):
        n_var, n = (500, 260) if i & 2 else (970, 90)
        kind = i // 2 % 4
        if kind < 2:
            made.append((*ancestry_panel(50 + i, n_var, n), n, 100, i & 1))
        elif kind == 2:
            made.append((*monomorphic_panel(50 + i, 970, 90, 60), 90, 300, i & 1))
        else:
            rng = np.random.default_rng(50 + i)
            planes = orc.planes_from_codes(orc.random_codes(rng, n_var, n, 0.01))
            made.append((*planes, *orc.masks_from_classes(rng.integers(0, 2, n)), n, 100, i & 1))
    items = [dict(panel=ge.Panel.from_planes(b, v, n), mask_ctrl=m0, mask_case=m1, topmost=k, ffun=f)
             for b, v, m0, m1, n, k, f in made]
    with ge.Engine() as eng:
        res, bs = eng.scan_batch(items)
    for i, ((b, v, m0, m1, n, k, f), (got, st, status)) in enumerate(zip(made, res)):
        assert status == 0
        assert_same(got, orc.gold_scan(orc.Panel(b, v, m0, m1, n), k, ffun=f), "item %d" % i)
        lost = st["pend_overflows"] + st["cand_overflows"]
        if i < 4:
            assert lost > 0, (i, st)                        # the guess was far too loose
        elif i < 6:
            assert lost == 0 and st["bands"] > 2, (i, st)   # too strict: begun again
        else:
            assert lost == 0 and st["bands"] <= 2, (i, st)
    assert bs["rounds"] <= 12, bs
    for it in items:
        it["panel"].close()


@pytest.mark.parametrize("n_var,n,k", [(300, 20000, 5000), (420, 46340, 20000)])
def test_fisher_many_samples(monkeypatch, n_var, n, k):
    """A table of many samples has a small probability whatever its p, so that
    the check of P(obs) passes nearly all evaluations under a loose threshold:
    no guess, in a single scan and batched."""
    print("case fisher many samples", n_var, n, k, flush=True)
    rng = np.random.default_rng(45)
    g = rng.integers(0, 2, (n_var, n)).astype(np.uint8) + (rng.random((n_var, n)) < 0.3)
    codes = np.array([3, 2, 0], np.uint8)[g]
    codes[::2][:, ::97] = 1
    bits, valid = orc.planes_from_codes(codes)
    m0, m1 = orc.masks_from_classes((rng.random(n) < 0.4).astype(int))
    with ge.Panel.from_planes(bits, valid, n) as panel:
        got, st = panel.scan(m0, m1, topmost=k, ffun=1)
        with ge.Engine() as eng:
            (res,), bs = eng.scan_batch([dict(panel=panel, mask_ctrl=m0, mask_case=m1, topmost=k, ffun=1)])
        ref, _ = band_by_band(monkeypatch, panel, m0, m1, k, 1, 20)
    assert_same(got, ref, "alone")
    assert_same(res[0], ref, "batch")
    assert st["bands"] <= 10 and bs["rounds"] <= 12, (st, bs)
