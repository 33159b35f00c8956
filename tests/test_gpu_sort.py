"""Long rankings: sorted on the device (tiles of 2,048 records, runs merged
pairwise) and, in scans much longer than the ranking, started under a guessed
threshold.  Against the oracle, and against the band-by-band loop without a
guess (a forced band size selects it)."""
import numpy as np
import pytest

import gepicount_amd as ge
from oracle import oracle as orc
from test_gpu_bands import associated_panel, band_by_band
from test_gpu_parity import assert_same, random_panel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [4096, 4097, 6144, 6145, 8191, 10241, 131073, 10 ** 6])
@pytest.mark.parametrize("noalloc", [False, True])
def test_sorted_on_device(k, noalloc):
    """One, an odd and an even number of tiles, last ones of one record and
    full ones; the last k holds every evaluation."""
    print("case device sort k=%d noalloc=%d" % (k, noalloc), flush=True)
    bits, valid, m0, m1 = random_panel(23, 150, 120, 0.02)
    with ge.Panel.from_planes(bits, valid, 120) as panel:
        scan = panel.scan_noalloc if noalloc else panel.scan
        got, _ = scan(m0, m1, topmost=k)
    ref = orc.gold_scan(orc.Panel(bits, valid, m0, m1, 120), k)
    assert len(got) == min(k, 5 * 150 * 301)
    assert_same(got, ref, "device-sort")


@pytest.mark.parametrize("ffun,path", [(0, 0), (1, 0), (0, 1), (0, 2)])
def test_long_ranking_starts_guessed(monkeypatch, ffun, path):
    print("case long ranking ffun=%d path=%d" % (ffun, path), flush=True)
    bits, valid, m0, m1 = random_panel(29, 3000, 200, 0.01)
    with ge.Panel.from_planes(bits, valid, 200) as panel:
        got, st = panel.scan(m0, m1, topmost=60000, ffun=ffun, count_path=path)
        ref, st_ref = band_by_band(monkeypatch, panel, m0, m1, 60000, ffun, 500)
    assert st["bands"] < st_ref["bands"]
    assert_same(got, ref, "long-ranking")


@pytest.mark.parametrize("ffun", [0, 1])
def test_long_ranking_guess_fails(monkeypatch, ffun):
    """Monomorphic but for every 40th variant: the guess admits fewer than k
    evaluations of the whole scan, which runs again without it."""
    print("case long ranking guess fails ffun=%d" % ffun, flush=True)
    rng = np.random.default_rng(31)
    codes = np.zeros((3000, 130), np.uint8)
    codes[::40] = rng.choice(np.array([0, 2, 3], np.uint8), size=codes[::40].shape)
    bits, valid = orc.planes_from_codes(codes)
    m0, m1 = orc.masks_from_classes(rng.integers(0, 2, 130))
    with ge.Panel.from_planes(bits, valid, 130) as panel:
        got, _ = panel.scan(m0, m1, topmost=60000, ffun=ffun)
        ref, _ = band_by_band(monkeypatch, panel, m0, m1, 60000, ffun, 500)
    assert_same(got, ref, "long-ranking-guess")


def test_long_ranking_overflow_is_redone():
    """Associated variants under the small lists of the allocation-free scan."""
    print("case long ranking overflow", flush=True)
    bits, valid, m0, m1 = associated_panel(7, 1200, 192)
    with ge.Panel.from_planes(bits, valid, 192) as panel:
        got, _ = panel.scan_noalloc(m0, m1, topmost=40000)
        ref, _ = panel.scan(m0, m1, topmost=40000)
    assert_same(got, ref, "long-ranking-overflow")
