"""The job shape of an autotuned engine: a class that keeps the default schedule
keeps its rule, by a scan's tiles and planes, which the trials' large panels on
genotype planes do not stand for.  Fewer than 256 tiles, and planes with a valid
call without an allele, against an engine without a table."""
import numpy as np
import pytest

import gepicount_amd as ge
from oracle import oracle as orc
from test_gpu_parity import assert_same
from test_gpu_screen import panel

pytestmark = pytest.mark.gpu


def test_default_classes_keep_their_rule(monkeypatch):
    print("case tuned shape", flush=True)
    monkeypatch.delenv("GEPI_F4_WG_PER_CU", raising=False)
    monkeypatch.delenv("GEPI_ENGINE_GRAPH", raising=False)
    made = [panel(130, 300, 60, 50, 0, 0.02), panel(131, 300, 400, 380, 0, 0.02),
            panel(132, 1000, 60, 50, 0, 0.02), panel(133, 1000, 60, 50, 0, 0.02)]
    bits, valid, m0, m1, n = made[3]
    bits = bits.copy()
    bits[0:2, 0] = 0
    made[3] = (bits, valid, m0, m1, n)
    items = [dict(panel=ge.Panel.from_planes(b, v, n), mask_ctrl=m0, mask_case=m1, topmost=100)
             for b, v, m0, m1, n in made]
    with ge.Engine() as eng:
        plain, _ = eng.scan_batch(items)
        table = eng.autotune(repeats=1)
        tuned, _ = eng.scan_batch(items)
        eng.set_tuning(table)
        again, _ = eng.scan_batch(items)
        # an explicit shape is the caller's for every scan of the class
        eng.set_tuning([dict(max_ksteps=2**31 - 1, wg_per_cu=2, tile=2, band_evals=2e9)])
        forced, _ = eng.scan_batch(items)
    print("table", table, flush=True)
    assert [r[1]["count_path"] for r in plain] == [4, 4, 3, 4]
    assert [r[1]["count_path"] for r in forced] == [3, 3, 3, 3]
    for i, (b, v, m0, m1, n) in enumerate(made):
        ref = orc.gold_scan(orc.Panel(b, v, m0, m1, n), 100)
        ks = sum(-(-int(np.bitwise_count(m).sum()) // 128) for m in (m0, m1))
        cls = next(c for c in table if ks <= c["max_ksteps"])
        for label, res in (("plain", plain), ("tuned", tuned), ("again", again), ("forced", forced)):
            assert_same(res[i][0], ref, "%s %d" % (label, i))
        if cls["tile"] == 2:  # wave tiles are the trials' default: kept, not chosen
            assert tuned[i][1]["count_path"] == plain[i][1]["count_path"], i
            assert again[i][1]["count_path"] == plain[i][1]["count_path"], i
    for it in items:
        it["panel"].close()
