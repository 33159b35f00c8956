"""Wave tiles on genotype planes: the screen of a pair's genotype table before
its 20 evaluations, the pairs collected per workgroup, and the class layout
made super-step by super-step.  Against the oracle at class sizes around the
384-sample super-steps and 32-bit words, with many missing calls, one empty
class, overlapping masks, more evaluations passing than a workgroup's list
holds, and a panel whose valid calls do not all carry an allele (which keeps
the allele planes)."""
import numpy as np
import pytest

import gepicount_amd as ge
from oracle import oracle as orc
from test_gpu_parity import assert_same

pytestmark = pytest.mark.gpu


def panel(seed, n_var, n0, n1, rest, miss):
    rng = np.random.default_rng(seed)
    n = n0 + n1 + rest
    codes = orc.random_codes(rng, n_var, n, miss)
    cls = np.full(n, -1)
    order = rng.permutation(n)
    cls[order[:n0]] = 0
    cls[order[n0:n0 + n1]] = 1
    bits, valid = orc.planes_from_codes(codes)
    m0, m1 = orc.masks_from_classes(cls)
    return bits, valid, m0, m1, n


@pytest.mark.parametrize("ffun", [0, 1])
@pytest.mark.parametrize("n_var,n0,n1,rest,miss,k", [
    (65, 383, 1, 0, 0.02, 300), (65, 384, 385, 7, 0.02, 300), (64, 31, 33, 0, 0.0, 500),
    (130, 769, 1152, 100, 0.3, 2000), (97, 0, 400, 3, 0.02, 100), (97, 400, 0, 3, 0.02, 100),
    (150, 1, 2, 0, 0.1, 50), (200, 96, 64, 40, 0.6, 5000), (33, 20, 500, 0, 0.9, 4000)])
def test_screen_equals_oracle(n_var, n0, n1, rest, miss, k, ffun):
    print("case screen", n_var, n0, n1, rest, miss, k, ffun, flush=True)
    bits, valid, m0, m1, n = panel(91, n_var, n0, n1, rest, miss)
    got, st = ge.process_gpu_1(bits, valid, m0, m1, n, topmost=k, ffun=ffun, count_path=3)
    assert st["count_path"] == 3
    assert_same(got, orc.gold_scan(orc.Panel(bits, valid, m0, m1, n), k, ffun=ffun), "screen")


@pytest.mark.parametrize("ffun", [0, 1])
def test_screen_list_overflow(monkeypatch, ffun):
    """A band under a loose threshold passes most pairs of a workgroup."""
    print("case screen overflow", ffun, flush=True)
    bits, valid, m0, m1, n = panel(92, 300, 200, 180, 0, 0.05)
    monkeypatch.setenv("GEPI_BAND_TILES", "3")
    got, _ = ge.process_gpu_1(bits, valid, m0, m1, n, topmost=40000, ffun=ffun, count_path=3)
    monkeypatch.delenv("GEPI_BAND_TILES")
    assert_same(got, orc.gold_scan(orc.Panel(bits, valid, m0, m1, n), 40000, ffun=ffun), "overflow")


@pytest.mark.parametrize("ffun", [0, 1])
def test_overlapping_masks(ffun):
    bits, valid, m0, m1, n = panel(93, 80, 300, 250, 50, 0.02)
    m1 = m1 | (m0 & np.uint64(0x0F0F0F0F0F0F0F0F))
    got, _ = ge.process_gpu_1(bits, valid, m0, m1, n, topmost=700, ffun=ffun, count_path=3)
    assert_same(got, orc.gold_scan(orc.Panel(bits, valid, m0, m1, n), 700, ffun=ffun), "overlap")


@pytest.mark.parametrize("ffun", [0, 1])
def test_valid_calls_without_an_allele(ffun):
    """Planes that no .bed file gives: a valid call with neither allele."""
    print("case neither allele", ffun, flush=True)
    bits, valid, m0, m1, n = panel(94, 90, 300, 280, 0, 0.02)
    rng = np.random.default_rng(95)
    drop = rng.integers(0, 2 ** 63, size=(90, bits.shape[1]), dtype=np.uint64) & \
        rng.integers(0, 2 ** 63, size=(90, bits.shape[1]), dtype=np.uint64)
    bits = bits & ~np.repeat(drop, 2, axis=0)
    got, st = ge.process_gpu_1(bits, valid, m0, m1, n, topmost=900, ffun=ffun, count_path=3)
    assert st["count_path"] == 3
    assert_same(got, orc.gold_scan(orc.Panel(bits, valid, m0, m1, n), 900, ffun=ffun), "neither")
