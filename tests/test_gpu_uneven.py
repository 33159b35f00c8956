"""Classes of very different size: scans that the screen of the genotype table
would hardly thin keep the allele planes (by the count path and, on wave tiles,
by the workspace: no list of put-off pairs).  Results against the oracle."""
import numpy as np
import pytest

import gepicount_amd as ge
from oracle import oracle as orc
from test_gpu_parity import assert_same
from test_gpu_screen import panel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_var,n0,n1,miss,k,ffun,path", [
    (970, 484, 28, 0.01, 100, 0, 4), (970, 484, 28, 0.0, 100, 0, 4), (970, 256, 256, 0.01, 100, 0, 3),
    (970, 410, 102, 0.0, 100, 0, 3), (970, 28, 484, 0.01, 100, 1, 4), (970, 1980, 68, 0.01, 100, 1, 3),
    (970, 1980, 68, 0.01, 100, 0, 3), (70, 2000, 3, 0.01, 300, 0, 3), (70, 3, 2000, 0.0, 300, 1, 3)])
def test_route(n_var, n0, n1, miss, k, ffun, path):
    print("case uneven", n_var, n0, n1, miss, k, ffun, flush=True)
    bits, valid, m0, m1, n = panel(140, n_var, n0, n1, 0, miss)
    ref = orc.gold_scan(orc.Panel(bits, valid, m0, m1, n), k, ffun=ffun)
    with ge.Panel.from_planes(bits, valid, n) as p:
        got, st = p.scan(m0, m1, topmost=k, ffun=ffun)
        assert_same(got, ref, "alone")
        assert st["count_path"] == path, st
        with ge.Engine() as eng:
            (res,), _ = eng.scan_batch([dict(panel=p, mask_ctrl=m0, mask_case=m1, topmost=k, ffun=ffun)])
        assert_same(res[0], ref, "batch")
        got, _ = p.scan_noalloc(m0, m1, topmost=k, ffun=ffun)
        assert_same(got, ref, "noalloc")
