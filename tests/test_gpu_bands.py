"""Planned bands: a scan enqueues all its bands at once under a threshold
guessed for the first one.  Their results against the band-by-band loop (a
forced band size selects it) and, where small enough, the oracle: a pilot
and the bands sized from it, lists that overflow, a guess that fails."""
import numpy as np
import pytest

import gepicount_amd as ge
from oracle import oracle as orc
from test_gpu_parity import assert_same, random_panel

pytestmark = pytest.mark.gpu


def band_by_band(monkeypatch, panel, m0, m1, k, ffun, tiles):
    monkeypatch.setenv("GEPI_BAND_TILES", str(tiles))
    ref, st = panel.scan(m0, m1, topmost=k, ffun=ffun)
    monkeypatch.delenv("GEPI_BAND_TILES")
    return ref, st


@pytest.mark.parametrize("n_var,n,k,ffun", [
    (700, 90, 1, 0), (700, 300, 3000, 0), (700, 300, 100, 1),  # the whole scan in one band
    (5200, 150, 100, 0), (5200, 150, 2500, 1),                 # a pilot, then the rest
    (5200, 1400, 20000, 0)])                                   # wave tiles, growing bands
def test_planned_equals_band_by_band(monkeypatch, n_var, n, k, ffun):
    print("case planned bands %d x %d top-%d ffun=%d" % (n_var, n, k, ffun), flush=True)
    bits, valid, m0, m1 = random_panel(71, n_var, n, 0.01)
    with ge.Panel.from_planes(bits, valid, n) as panel:
        got, st = panel.scan(m0, m1, topmost=k, ffun=ffun)
        ref, st_ref = band_by_band(monkeypatch, panel, m0, m1, k, ffun, 64)
    assert st["bands"] < st_ref["bands"]
    assert_same(got, ref, "planned")


def associated_panel(seed, n_var, n):
    """Variants that follow the phenotype for a part of the samples, so that
    far more evaluations pass any threshold than by chance."""
    rng = np.random.default_rng(seed)
    cls = rng.integers(0, 2, n)
    codes = rng.choice(np.array([0, 2, 3], np.uint8), size=(n_var, n))
    follow = rng.random((n_var, n)) < 0.35
    codes[follow] = np.broadcast_to(np.where(cls == 1, 0, 3).astype(np.uint8), (n_var, n))[follow]
    bits, valid = orc.planes_from_codes(codes)
    m0, m1 = orc.masks_from_classes(cls)
    return bits, valid, m0, m1


@pytest.mark.parametrize("ffun", [0, 1])
def test_planned_overflow_is_redone(ffun):
    """The allocation-free scan's lists hold about 83,000 records more than
    k: here most evaluations pass the guessed threshold, and the band is
    redone in pieces."""
    print("case planned overflow ffun=%d" % ffun, flush=True)
    bits, valid, m0, m1 = associated_panel(5, 400, 256)
    with ge.Panel.from_planes(bits, valid, 256) as panel:
        got, st = panel.scan_noalloc(m0, m1, topmost=200, ffun=ffun)
    assert st["pend_overflows"] + st["cand_overflows"] > 0
    ref = orc.gold_scan(orc.Panel(bits, valid, m0, m1, 256), 200, ffun=ffun)
    assert_same(got, ref, "planned-overflow")


@pytest.mark.parametrize("ffun", [0, 1])
def test_planned_guess_fails(ffun):
    """All but 60 of 400 variants are monomorphic: fewer than k evaluations
    reach the guessed threshold, and the scan is run again without it."""
    print("case planned guess fails ffun=%d" % ffun, flush=True)
    rng = np.random.default_rng(9)
    codes = np.zeros((400, 130), np.uint8)
    codes[::7] = rng.choice(np.array([0, 2, 3], np.uint8), size=codes[::7].shape)
    bits, valid = orc.planes_from_codes(codes)
    m0, m1 = orc.masks_from_classes(rng.integers(0, 2, 130))
    got, st = ge.process_gpu_1(bits, valid, m0, m1, 130, topmost=1500, ffun=ffun)
    ref = orc.gold_scan(orc.Panel(bits, valid, m0, m1, 130), 1500, ffun=ffun)
    assert_same(got, ref, "planned-guess")


@pytest.mark.parametrize("n_var,n,k", [(1, 40, 3), (2, 50, 10), (20, 300, 1000), (64, 100, 2000)])
@pytest.mark.parametrize("ffun", [0, 1])
def test_tiny_panels(n_var, n, k, ffun):
    """A tile of these holds a fraction of a whole tile's evaluations: no guess
    for a ranking of much of the panel, and not a band that is lost."""
    print("case tiny", n_var, n, k, ffun, flush=True)
    bits, valid, m0, m1 = random_panel(73, n_var, n, 0.01)
    with ge.Panel.from_planes(bits, valid, n) as panel:
        got, st = panel.scan(m0, m1, topmost=k, ffun=ffun)
    assert st["bands"] <= 2, st
    assert_same(got, orc.gold_scan(orc.Panel(bits, valid, m0, m1, n), k, ffun=ffun), "tiny")


@pytest.mark.parametrize("ffun", [0, 1])
def test_long_bands(monkeypatch, ffun):
    """No planned band of a long scan is much more than a third of it: what
    one that turns out to pass too much has cost is small."""
    print("case long bands ffun=%d" % ffun, flush=True)
    rng = np.random.default_rng(75)
    byte = np.array([a | b << 2 | c << 4 | d << 6 for a in (0, 2, 3) for b in (0, 2, 3) for c in (0, 2, 3) for d in (0, 2, 3)], np.uint8)
    n_var, n = 40000, 4096
    payload = byte[rng.integers(0, 81, (n_var, n // 4), np.uint8)]
    m0, m1 = orc.masks_from_classes(rng.integers(0, 2, n))
    with ge.Panel.from_bed(payload, n_var, n) as panel:
        got, st = panel.scan(m0, m1, topmost=100, ffun=ffun)
        ref, _ = band_by_band(monkeypatch, panel, m0, m1, 100, ffun, 65536)
    assert st["bands"] >= 6, st
    assert_same(got, ref, "long bands")


def test_batch_guess_too_strict():
    """With 8 cases few tables are as improbable as the guess assumes: the
    scans of a batch go on under a looser one, not from a single tile."""
    print("case batch guess too strict", flush=True)
    rng = np.random.default_rng(77)
    codes = np.array([0, 2, 3], np.uint8)
    items, refs = [], []
    for j in range(4):
        f = rng.uniform(0.05, 0.5, (3000, 1, 1))
        dose = (rng.random((3000, 400, 2)) < f).sum(2)
        bits, valid = orc.planes_from_codes(codes[dose])
        cls = np.zeros(400, np.int64)
        cls[rng.choice(400, 8, replace=False)] = 1
        m0, m1 = orc.masks_from_classes(cls)
        items.append(dict(panel=ge.Panel.from_planes(bits, valid, 400), mask_ctrl=m0, mask_case=m1, topmost=100, ffun=1))
        refs.append(items[-1]["panel"].scan(m0, m1, topmost=100, ffun=1)[0])
    eng = ge.Engine()
    res, bs = eng.scan_batch(items)
    eng.close()
    for j in range(4):
        items[j]["panel"].close()
        assert_same(res[j][0], refs[j], "batch %d" % j)
    assert bs["rounds"] <= 4, bs
