"""The product-count scan (scan.hip) through brm_flop_count_dev, against
numpy: lengths at and around one wavefront, one tile of 1,024 or 2,048
elements, the most tiles that every block adds up for itself, and beyond;
counts of a few entries and of almost 2^31."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LEN = [0, 1, 63, 65, 1023, 1024, 1025, 524288, 524289, 526337, 8192 * 2048, 8192 * 2048 + 1, 8192 * 2048 + 2049]


@pytest.mark.parametrize("big", [False, True])
@pytest.mark.parametrize("n", LEN)
def test_product_counts(gpu, n, big):
    bm = gpu
    L = bm.lib()
    rng = np.random.default_rng(n + big)
    K = 1000
    if big:  # one row of almost 2^31 entries among empty ones (only the row pointer is read)
        brpt = np.zeros(K + 1, np.int32)
        brpt[501:] = 2 ** 31 - 2
    else:
        brpt = np.concatenate([[0], np.cumsum(rng.integers(0, 30, K))]).astype(np.int32)
    acol = rng.integers(0, K, n).astype(np.int32)
    if big and n:
        acol[rng.integers(0, n, 3)] = 500
    # rows of A: cuts at random places
    M = 50
    arpt = np.concatenate([[0], np.sort(rng.integers(0, n + 1, M - 1)), [n]]).astype(np.int32)
    ip = np.concatenate([[0], np.cumsum(np.diff(brpt.astype(np.int64))[acol])])
    dev = [bm.DeviceArray.from_host(x) for x in (arpt, acol, brpt)]
    rows = bm.DeviceArray.alloc(M, np.int64)
    tot = ctypes.c_int64()
    try:
        for _ in range(2):
            assert L.brm_flop_count_dev(dev[0].ptr, dev[1].ptr, n, dev[2].ptr, M, K, rows.ptr, ctypes.byref(tot), None) == 0
            assert tot.value == ip[-1]
            np.testing.assert_array_equal(rows.to_host(), ip[arpt[1:]] - ip[arpt[:-1]])
    finally:
        for d in dev + [rows]:
            d.free()
