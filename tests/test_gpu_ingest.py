"""Decoding of .bed payloads and missing-call counts at the edges of their
blocks: rows that start at any byte, samples around 64 and 4,096, variants
around the 7 words added at a time, the 112 of a wave and the 448 of a block.
Against numpy, identical."""
import numpy as np
import pytest

import gepicount_amd as ge

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_var,n", [(1, 1), (7, 3), (8, 64), (111, 65), (112, 5), (113, 130),
                                     (448, 71), (449, 4096), (900, 4097), (33, 8200)])
def test_decode_and_counts(n_var, n):
    print("case ingest", n_var, n, flush=True)
    rng = np.random.default_rng(n_var * 10007 + n)
    n4 = (n + 3) // 4
    payload = rng.integers(0, 256, size=(n_var, n4), dtype=np.uint8)  # padding codes set too
    codes = ((payload[:, :, None] >> np.array([0, 2, 4, 6])) & 3).reshape(n_var, 4 * n4)[:, :n]
    p = ge.Panel.from_bed(payload, n_var, n)
    bits, valid = p.download()
    w = (n + 63) // 64

    def plane(m):
        full = np.zeros((n_var, 64 * w), np.uint8)
        full[:, :n] = m
        return np.packbits(full, axis=1, bitorder="little").view(np.uint64)

    assert np.array_equal(bits[0::2], plane((codes == 0) | (codes == 2)))
    assert np.array_equal(bits[1::2], plane((codes == 2) | (codes == 3)))
    assert np.array_equal(valid[0::2], plane(codes != 1))
    vm, sm, _, _ = p.qa()
    assert np.array_equal(vm, (codes == 1).sum(1))
    assert np.array_equal(sm, (codes == 1).sum(0))
    p.close()
