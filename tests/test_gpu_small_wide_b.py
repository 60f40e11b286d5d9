"""The fused short-row path with many more rows in B than in A (a few rows of
A naming rows of a large B): B's rows at and around what its checking
workgroups take in one turn, in groups of 32 and of 64 lanes; faults in the
first, a middle and the last row are found; and it takes no longer than the
general pipeline."""
import time

import numpy as np
import pytest

import oracle
from tests._util import assert_csr_equal, csr_from_tuple

pytestmark = pytest.mark.gpu

TURN = {32: 2048 * 512, 64: 2048 * 1024}  # rows of B


def _operands(rng, K, group, M=100):
    per, N = (5, 5000) if group == 32 else (8, 5000)
    c = np.sort(rng.integers(0, N - per, (K, per)), axis=1) + np.arange(per)
    acol = np.sort(rng.choice(K, (M, per), replace=False), axis=1)
    acol[0, 0], acol[-1, -1] = 0, K - 1
    A = (np.arange(M + 1, dtype=np.int32) * per, acol.reshape(-1).astype(np.int32), rng.uniform(-1, 1, M * per), K)
    B = (np.arange(K + 1, dtype=np.int32) * per, c.reshape(-1).astype(np.int32), rng.uniform(-1, 1, K * per), N)
    return A, B, per


@pytest.mark.parametrize("group", [32, 64])
@pytest.mark.parametrize("more", [-2, -1, 0, 1, 513, 3 * 10 ** 6])
def test_rows_of_b(gpu, group, more):
    bm = gpu
    rng = np.random.default_rng(group + more + 10)
    K = TURN[group] + more
    A, B, per = _operands(rng, K, group)
    R = oracle.brmerge_precise(A, B, nthreads=4)
    dA = bm.DeviceCSR.upload(csr_from_tuple(A))

    def product(T):
        dB = bm.DeviceCSR.upload(csr_from_tuple(T))
        try:
            C = bm.spgemm_dev(dA, dB)
            H = C.download()
            C.free()
            return H
        finally:
            dB.free()

    assert_csr_equal(product(B), R)
    for row in (0, K // 2, K - 1):
        col = B[1].copy()
        col[row * per:row * per + 2] = col[row * per:row * per + 2][::-1]
        with pytest.raises(bm.BrmError) as e:
            product((B[0], col, B[2], B[3]))
        assert e.value.status == 1
    rpt = B[0].copy()
    rpt[0] = 1
    with pytest.raises(bm.BrmError) as e:  # the row pointer begins past the first entry
        product((rpt, B[1], B[2], B[3]))
    assert e.value.status == 1
    dA.free()


def test_time(gpu):
    bm = gpu
    rng = np.random.default_rng(2)
    K, M = 2 * 10 ** 7, 2048
    A = bm.CSR(np.arange(M + 1, dtype=np.int32) * 4, np.sort(rng.integers(0, K // 4, (M, 4)) * 4 + np.arange(4), axis=1).reshape(-1).astype(np.int32),
               np.ones(4 * M), M, K)
    B = bm.CSR(np.arange(K + 1, dtype=np.int32), rng.integers(0, 10 ** 6, K).astype(np.int32), np.ones(K), K, 10 ** 6)
    dA, dB = bm.DeviceCSR.upload(A), bm.DeviceCSR.upload(B)
    old = bm.get_param("small_fused")
    best = {}
    try:
        for fused in (0, 1):
            bm.set_param("small_fused", fused)
            t = []
            for _ in range(9):
                t0 = time.perf_counter()
                bm.spgemm_dev(dA, dB).free()
                t.append(time.perf_counter() - t0)
            best[fused] = min(t)
    finally:
        bm.set_param("small_fused", old)
        dA.free()
        dB.free()
    assert best[1] < best[0], best
