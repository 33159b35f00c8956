"""The automatic choice between the wave tiles and the LDS-staged kernel on
both sides of its lines: entropy at 256 tiles, Fisher at its evaluations per
record.  Results against the oracle, identical."""
import pytest

import gepicount_amd as ge
from oracle import oracle as orc
from test_gpu_parity import assert_same
from test_gpu_screen import panel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_var,n0,n1,miss,k,ffun,path", [
    (960, 60, 40, 0.02, 200, 0, 4), (961, 60, 40, 0.02, 200, 0, 3), (961, 60, 40, 0.0, 200, 0, 3),
    (961, 640, 641, 0.02, 10, 1, 3), (961, 640, 641, 0.02, 12, 1, 4), (961, 640, 641, 0.0, 12, 1, 3),
    (961, 640, 641, 0.0, 24, 1, 4)])
def test_route(n_var, n0, n1, miss, k, ffun, path):
    print("case route", n_var, n0, n1, miss, k, ffun, flush=True)
    bits, valid, m0, m1, n = panel(110, n_var, n0, n1, 0, miss)
    got, st = ge.process_gpu_1(bits, valid, m0, m1, n, topmost=k, ffun=ffun)
    assert st["count_path"] == path
    assert_same(got, orc.gold_scan(orc.Panel(bits, valid, m0, m1, n), k, ffun=ffun), "route")
