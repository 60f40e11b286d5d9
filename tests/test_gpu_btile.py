"""GPU parity of the column-tile long-row engine (btile.hip) against the
oracle, bit for bit, at block counts from 2 (every block too full for a round,
cut by column searches) to 4,096 (more blocks than columns): rows dense over a
few thousand columns, rows of thousands of lists with hub columns (three
passes, node tables read by the next pass), columns spread over 2^31 - 1
(rounds bounded by their column span), single lists, empty lists, and several
workspace waves on two streams."""
import numpy as np
import pytest

import oracle
from tests._util import assert_csr_equal, csr_from_tuple

pytestmark = pytest.mark.gpu


def _csr(rows, N, rng):
    rpt = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    col = np.concatenate(rows).astype(np.int32)
    return rpt, col, rng.uniform(-1, 1, len(col)) * rng.choice([1.0, 2.0 ** 30, 2.0 ** -30, 0.0], len(col)), N


def _case(name, rng):
    if name == "dense":  # 100 lists, each all of 3,000 columns but a few
        N = 3000
        B = [np.sort(rng.choice(N, N - int(rng.integers(0, 9)), replace=False)) for _ in range(100)]
        A = [np.arange(100), np.sort(rng.choice(100, 64, replace=False)), np.array([7])]
    elif name == "hubs":  # 5,000 lists of 1 to 30 columns, most of them through two hubs
        N = 20000
        B = [np.unique(np.concatenate([[17, 9001][:int(rng.integers(0, 3))], rng.integers(0, N, int(rng.integers(1, 31)))]))
             for _ in range(5000)]
        A = [np.arange(5000), np.sort(rng.choice(5000, 4097, replace=False)), np.sort(rng.choice(5000, 65, replace=False))]
    elif name == "wide":  # lists over 2^31 - 1 columns, both ends included
        N = (1 << 31) - 1
        B = [np.unique(np.concatenate([[0, N - 1], rng.integers(0, N, 200)])) for _ in range(70)]
        A = [np.arange(70), np.arange(33), np.array([1])]
    elif name == "edges":  # columns at the edges of 2^16-column spans
        N = 5 << 16
        e = np.arange(1, 5) << 16
        pool = np.unique(np.concatenate([e - 1, e, e + 1, [0, N - 1], rng.integers(0, N, 3000)]))
        B = [np.sort(rng.choice(pool, int(rng.integers(100, 900)), replace=False)) for _ in range(130)]
        A = [np.arange(130), np.arange(64), np.arange(65)]
    else:  # empty lists among lists of one to three columns
        N = 400
        B = [np.sort(rng.choice(N, int(rng.integers(0, 4)), replace=False)) for _ in range(9000)]
        A = [np.arange(9000), np.arange(0, 9000, 3), np.arange(64)]
    return _csr(A, len(B), rng), _csr(B, N, rng)


@pytest.mark.parametrize("blocks", [2, 64, 1024, 4096])
@pytest.mark.parametrize("case", ["dense", "hubs", "wide", "edges", "empty"])
def test_tiles(gpu, case, blocks):
    bm = gpu
    rng = np.random.default_rng(len(case) * 7 + blocks)
    A, B = _case(case, rng)
    R = oracle.brmerge_precise(A, B, nthreads=4)
    Ah, Bh = csr_from_tuple(A), csr_from_tuple(B)
    saved = {k: bm.get_param(k) for k in ("force_long", "long_tiles", "ws_budget_bytes")}
    try:
        bm.set_param("force_long", 1)
        bm.set_param("long_tiles", blocks)
        for ws in (0, 1 << 16):  # one wave, one row per wave
            bm.set_param("ws_budget_bytes", ws)
            for f in (bm.brmerge_precise, bm.brmerge_upper):
                assert_csr_equal(f(Ah, Bh), R)
    finally:
        for k, v in saved.items():
            bm.set_param(k, v)
