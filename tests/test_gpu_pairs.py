"""Pairs that pass the screen and are put off to a launch of their own
(k_pairs): more of them than the list holds (the rest is tested in the count
kernel), class sizes on both sides of the rule's 48 K steps, and the batch
engine's form.  Against the oracle, every field identical."""
import numpy as np
import pytest

import gepicount_amd as ge
from oracle import oracle as orc
from test_gpu_parity import assert_same
from test_gpu_screen import panel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ffun", [0, 1])
def test_more_pairs_than_the_list(monkeypatch, ffun):
    """260 variants in one band that admits everything: 33,930 pairs, a list of 15,360."""
    print("case pairs overflow", ffun, flush=True)
    bits, valid, m0, m1, n = panel(96, 260, 90, 70, 0, 0.03)
    monkeypatch.setenv("GEPI_BAND_TILES", "64")
    got, _ = ge.process_gpu_1(bits, valid, m0, m1, n, topmost=20000, ffun=ffun, count_path=3)
    monkeypatch.delenv("GEPI_BAND_TILES")
    assert_same(got, orc.gold_scan(orc.Panel(bits, valid, m0, m1, n), 20000, ffun=ffun), "list")


@pytest.mark.parametrize("ffun", [0, 1])
@pytest.mark.parametrize("n0,n1", [(3072, 3072), (3073, 3072)])
def test_both_sides_of_the_rule(n0, n1, ffun):
    print("case pairs rule", n0, n1, ffun, flush=True)
    bits, valid, m0, m1, n = panel(97, 66, n0, n1, 0, 0.02)
    got, _ = ge.process_gpu_1(bits, valid, m0, m1, n, topmost=400, ffun=ffun, count_path=3)
    assert_same(got, orc.gold_scan(orc.Panel(bits, valid, m0, m1, n), 400, ffun=ffun), "rule")


def test_batch():
    """Both objectives in one batch, scans long enough for genotype planes."""
    print("case pairs batch", flush=True)
    made, items = [], []
    for i, (n_var, k) in enumerate([(970, 300), (1000, 20), (990, 100)]):
        bits, valid, m0, m1, n = panel(98 + i, n_var, 40, 35, 2, 0.02)
        made.append((bits, valid, m0, m1, n, k, i & 1))
        items.append(dict(panel=ge.Panel.from_planes(bits, valid, n), mask_ctrl=m0, mask_case=m1, topmost=k, ffun=i & 1))
    eng = ge.Engine()
    res, _ = eng.scan_batch(items)
    for (bits, valid, m0, m1, n, k, ffun), (got, _, status) in zip(made, res):
        assert status == 0
        assert_same(got, orc.gold_scan(orc.Panel(bits, valid, m0, m1, n), k, ffun=ffun), "batch")
    eng.close()
