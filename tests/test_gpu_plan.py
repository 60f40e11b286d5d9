"""The long-row planner (k_plan_small, k_plan_large) against the oracle, bit
for bit: rows of 1 to 64 lists (one wavefront), of 65 and more (several
workgroups), of two and three passes, at the edges of a step's nodes; empty
rows, empty lists, rows of empty lists only; whole launches and launches of
three rows; with and without the block tables."""
import numpy as np
import pytest

import oracle
from tests._util import assert_csr_equal, csr_from_tuple

pytestmark = pytest.mark.gpu

LENS = [0, 1, 2, 63, 64, 65, 127, 128, 129, 255, 256, 257, 300, 1024, 4095, 4096, 4097, 4160, 8193]


@pytest.mark.parametrize("chunk", [0, 3])
@pytest.mark.parametrize("tiles", [0, 64])
@pytest.mark.parametrize("empty", [0.0, 0.6])
def test_planned_rows(gpu, chunk, tiles, empty):
    bm = gpu
    rng = np.random.default_rng(int(10 * empty) + chunk + tiles)
    K, N = 8500, 5000
    blen = np.where(rng.random(K) < empty, 0, rng.integers(1, 5, K))
    blen[:100] = 0
    brows = [np.sort(rng.choice(N, n, replace=False)) for n in blen]
    rows = [np.sort(rng.choice(K, n, replace=False)) for n in LENS]
    rows += [np.arange(70), np.arange(30)]  # of empty lists only
    rows = [rows[i] for i in rng.permutation(len(rows))]

    def csr(rr, ncol):
        rpt = np.concatenate([[0], np.cumsum([len(r) for r in rr])]).astype(np.int32)
        col = np.concatenate(rr).astype(np.int32)
        return rpt, col, rng.uniform(-1, 1, len(col)) * rng.choice([1.0, 2.0 ** 40, 0.0], len(col)), ncol

    A, B = csr(rows, K), csr(brows, N)
    R = oracle.brmerge_precise(A, B, nthreads=4)
    Ah, Bh = csr_from_tuple(A), csr_from_tuple(B)
    names = ("force_long", "long_tiles", "launch_chunk", "ws_budget_bytes")
    saved = {k: bm.get_param(k) for k in names}
    try:
        bm.set_param("force_long", 1)
        bm.set_param("long_tiles", tiles)
        bm.set_param("launch_chunk", chunk)
        for ws in (0, 1 << 17):
            bm.set_param("ws_budget_bytes", ws)
            for f in (bm.brmerge_precise, bm.brmerge_upper):
                assert_csr_equal(f(Ah, Bh), R)
    finally:
        for k, v in saved.items():
            bm.set_param(k, v)
