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


@pytest.mark.parametrize("cap", ["0", "100"])
def test_list_left_out(monkeypatch, cap):
    """No list, as where it does not fit, and a short one: single scans, the engine
    and a server whose budget leaves no room for it."""
    print("case pairs left out", cap, flush=True)
    monkeypatch.setenv("GEPI_PAIR_CAP", cap)
    made = [panel(120 + i, 970 + i, 40, 35, 2, 0.02) for i in range(2)]
    refs = [orc.gold_scan(orc.Panel(b, v, m0, m1, n), 200, ffun=i) for i, (b, v, m0, m1, n) in enumerate(made)]
    ps = [ge.Panel.from_planes(b, v, n) for b, v, _, _, n in made]
    for i, (p, (_, _, m0, m1, _)) in enumerate(zip(ps, made)):
        got, _ = p.scan(m0, m1, topmost=200, ffun=i, count_path=3)
        assert_same(got, refs[i], "alone")
    with ge.Engine() as eng:
        res, _ = eng.scan_batch([dict(panel=p, mask_ctrl=m0, mask_case=m1, topmost=200, ffun=i)
                                 for i, (p, (_, _, m0, m1, _)) in enumerate(zip(ps, made))])
    for r, ref in zip(res, refs):
        assert_same(r[0], ref, "batch")
    for p in ps:
        p.close()


def test_list_does_not_count_against_the_budget():
    """Requests are admitted by what they cannot do without: while a large scan
    runs, ten of about 31 MB each join it under a budget that holds them (and
    two of them with their lists of pairs, 101 MB each)."""
    print("case pairs budget", flush=True)
    rng = np.random.default_rng(7)

    def bed(n_var, n):
        m0, m1 = orc.masks_from_classes(rng.integers(0, 2, n))
        return rng.integers(0, 256, size=(n_var, (n + 3) // 4), dtype=np.uint8), n_var, n, m0, m1

    large, small = bed(50000, 4000), [bed(20000, 256) for _ in range(10)]
    with ge.Server(hbm_budget=560 << 20) as srv:
        ids = [srv.add_panel_bed(*x[:3]) for x in [large] + small]
        asks = [(i, x[3], x[4]) for i, x in zip(ids, [large] + small)]
        tickets = [srv.submit(i, m0, m1, topmost=100) for i, m0, m1 in asks]
        res = [srv.wait(t) for t in tickets]
        st = srv.stats()
    assert st["failed"] == 0
    assert st["max_active"] >= 8, st
    for (got, _, status), x in zip(res[1:4], small):
        assert status == 0
        with ge.Panel.from_bed(*x[:3]) as p:
            assert_same(got, p.scan(x[3], x[4], topmost=100)[0], "served")
