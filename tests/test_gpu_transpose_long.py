"""The device transpose with rows too long for the lanes that the average row
gets: rows at and around the length from which they are written in pieces and
around multiples of it, beginning at, before and after an entry where a piece
begins, first, last and next to each other, among rows of few entries or none.
And its time: a matrix with one row of 10^6 entries takes at most 3 times as
long as one of as many entries in even rows."""
import time

import numpy as np
import pytest

from tests._util import assert_csr_equal

pytestmark = pytest.mark.gpu

LONG = [511, 512, 513, 1023, 1024, 1025, 1536, 40000]


def _matrix(rng, lens, N):
    rpt = np.concatenate([[0], np.cumsum(lens)])
    col = rng.integers(0, N, rpt[-1])
    for i in np.flatnonzero(np.asarray(lens) > 1):
        col[rpt[i]:rpt[i + 1]] = np.sort(rng.choice(N, lens[i], replace=False))
    return rpt.astype(np.int32), col.astype(np.int32)


@pytest.mark.parametrize("where", ["apart", "together", "alone"])
@pytest.mark.parametrize("few", [1, 6, 20, 60])  # 1, 4, 16 and 64 lanes per row
@pytest.mark.parametrize("shift", [0, 1, 511])
def test_long_rows(gpu, few, shift, where):
    bm = gpu
    rng = np.random.default_rng(few + shift + len(where))
    N = 50000
    if where == "alone":
        lens = [shift, 40000]
    elif where == "together":
        lens = [shift] + LONG + [few] * 100000
    else:
        lens = [shift]
        for n in LONG:
            lens += [n, 0, 0] + [few] * 10000 + [0]
        lens += [513]
    lens = np.asarray(lens)
    rpt, col = _matrix(rng, lens, N)
    A = bm.CSR(rpt, col, rng.uniform(-1, 1, len(col)), len(lens), N)
    dA = bm.DeviceCSR.upload(A)
    dT = dA.transpose()
    assert_csr_equal(dT.download(), A.transpose())
    dA.free()
    dT.free()


def test_time_of_one_long_row(gpu):
    bm = gpu
    rng = np.random.default_rng(1)
    M = 1000000
    best = []
    for hub in (1, M):
        lens = np.ones(M, np.int64)
        lens[M // 2] = hub
        if hub == 1:
            lens[:] = 2
        rpt = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
        col = rng.integers(0, M, rpt[-1]).astype(np.int32)
        dA = bm.DeviceCSR.upload(bm.CSR(rpt, col, np.ones(len(col)), M, M))
        t = []
        for _ in range(5):
            t0 = time.perf_counter()
            dA.transpose().free()
            t.append(time.perf_counter() - t0)
        best.append(min(t))
        dA.free()
    assert best[1] < 3 * best[0], best
