"""Panels without missing calls: four products a pair, the other cells from the
variants' own counts.  Class sizes around the 384-sample super-steps, one empty
class, overlapping masks, samples of neither class, rare genotypes, both ways a
panel is made, the list's overflow and the batch engine; a panel with a single
missing call keeps the nine products.  Against the oracle, identical."""
import numpy as np
import pytest

import gepicount_amd as ge
from oracle import oracle as orc
from test_gpu_parity import assert_same
from test_gpu_screen import panel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ffun", [0, 1])
@pytest.mark.parametrize("n_var,n0,n1,rest,k", [
    (1, 5, 6, 0, 15), (65, 383, 1, 0, 300), (64, 384, 385, 7, 300), (130, 769, 1152, 100, 2000),
    (97, 0, 400, 3, 100), (97, 400, 0, 3, 100), (150, 1, 2, 0, 50), (33, 3073, 3080, 1, 400)])
def test_complete_equals_oracle(n_var, n0, n1, rest, k, ffun):
    print("case complete", n_var, n0, n1, rest, k, ffun, flush=True)
    bits, valid, m0, m1, n = panel(101, n_var, n0, n1, rest, 0.0)
    ref = orc.gold_scan(orc.Panel(bits, valid, m0, m1, n), k, ffun=ffun)
    got, st = ge.process_gpu_1(bits, valid, m0, m1, n, topmost=k, ffun=ffun, count_path=3)
    assert st["count_path"] == 3
    assert_same(got, ref, "planes")


@pytest.mark.parametrize("lost", [0, 1])
@pytest.mark.parametrize("ffun", [0, 1])
def test_bed_panels(ffun, lost):
    """Rare alleles (most cells empty); the same with one call missing."""
    print("case complete bed", ffun, lost, flush=True)
    rng = np.random.default_rng(102)
    n_var, n = 90, 501
    g = (rng.random((n_var, n)) < 0.03).astype(np.uint8) + (rng.random((n_var, n)) < 0.03)
    codes = np.array([3, 2, 0], np.uint8)[g]
    if lost:
        codes[89, 500] = 1
    c = np.zeros((n_var, 504), np.uint8)
    c[:, :n] = codes
    c = c.reshape(n_var, 126, 4)
    payload = c[:, :, 0] | (c[:, :, 1] << 2) | (c[:, :, 2] << 4) | (c[:, :, 3] << 6)
    cls = rng.choice([0, 1, -1], size=n, p=[0.5, 0.4, 0.1])
    m0, m1 = orc.masks_from_classes(cls)
    m1 = m1 | (m0 & np.uint64(0x0F0F0F0F0F0F0F0F))  # some in both classes
    bits, valid = orc.planes_from_codes(codes)
    p = ge.Panel.from_bed(payload, n_var, n)
    got, _ = p.scan(m0, m1, topmost=3000, ffun=ffun, count_path=3)
    assert_same(got, orc.gold_scan(orc.Panel(bits, valid, m0, m1, n), 3000, ffun=ffun), "bed")
    kept, idx, _ = p.filter()
    got, _ = kept.scan(m0, m1, topmost=3000, ffun=ffun, count_path=3)
    assert len(idx) == n_var
    assert_same(got, orc.gold_scan(orc.Panel(bits, valid, m0, m1, n), 3000, ffun=ffun), "filtered")
    kept.close()
    p.close()


@pytest.mark.parametrize("ffun", [0, 1])
def test_list_overflow(monkeypatch, ffun):
    print("case complete overflow", ffun, flush=True)
    bits, valid, m0, m1, n = panel(103, 260, 90, 70, 0, 0.0)
    monkeypatch.setenv("GEPI_BAND_TILES", "64")
    got, _ = ge.process_gpu_1(bits, valid, m0, m1, n, topmost=20000, ffun=ffun, count_path=3)
    monkeypatch.delenv("GEPI_BAND_TILES")
    assert_same(got, orc.gold_scan(orc.Panel(bits, valid, m0, m1, n), 20000, ffun=ffun), "list")


def test_batch():
    """Both objectives, with and without missing calls, in one batch."""
    print("case complete batch", flush=True)
    made, items = [], []
    for i in range(4):
        bits, valid, m0, m1, n = panel(104 + i, 970 + i, 40, 35, 2, 0.02 if i > 1 else 0.0)
        made.append((bits, valid, m0, m1, n, i & 1))
        items.append(dict(panel=ge.Panel.from_planes(bits, valid, n), mask_ctrl=m0, mask_case=m1,
                          topmost=200, ffun=i & 1))
    eng = ge.Engine()
    res, _ = eng.scan_batch(items)
    for (bits, valid, m0, m1, n, ffun), (got, _, status) in zip(made, res):
        assert status == 0
        assert_same(got, orc.gold_scan(orc.Panel(bits, valid, m0, m1, n), 200, ffun=ffun), "batch")
    eng.close()


@pytest.mark.parametrize("ffun", [0, 1])
def test_without_allocation(ffun):
    """The margins lie in the scan's fixed scratch there, and no list is kept."""
    print("case complete noalloc", ffun, flush=True)
    bits, valid, m0, m1, n = panel(109, 100, 700, 650, 3, 0.0)
    p = ge.Panel.from_planes(bits, valid, n)
    got, _ = p.scan_noalloc(m0, m1, topmost=600, ffun=ffun, count_path=3)
    assert_same(got, orc.gold_scan(orc.Panel(bits, valid, m0, m1, n), 600, ffun=ffun), "noalloc")
    p.close()
