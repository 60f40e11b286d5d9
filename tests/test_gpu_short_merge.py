"""GPU parity of the short rows' register merge (short_merge.h) and of the
fused path's workgroup shapes (small.hip) against the oracle, bit for bit:
row counts at which the number of passes changes and at which the last
workgroup is full, one row short or one row over; columns that fit the packed
sort keys and columns that do not; rows whose lists all meet in one column (a
tree of all levels), whose lists are of very different lengths, some of them
empty; signed zeros."""
import numpy as np
import pytest

import oracle
from tests._util import assert_csr_equal, csr_from_tuple

pytestmark = pytest.mark.gpu


def _operands(rng, M, N, group):
    K = 300
    # B: lists of 0 to 5 entries, mostly through one hub column
    hub = int(rng.integers(0, N))
    blen = rng.choice([0, 1, 1, 2, 3, 5], size=K)
    brows = [np.unique(np.concatenate([[hub] if rng.random() < 0.8 else [], rng.integers(0, N, int(n))])).astype(np.int64)[:int(n)]
             for n in blen]
    blen = np.array([len(r) for r in brows])
    brpt = np.concatenate([[0], np.cumsum(blen)]).astype(np.int32)
    bcol = np.concatenate(brows).astype(np.int32)
    pool = [np.sort(rng.permutation(K)[:int(n)]) for n in rng.integers(0, group + 1, size=64)]
    pool.append(np.flatnonzero(blen == 1)[:group])  # as many lists as lanes
    for i, p in enumerate(pool):  # at most `group` products in a row
        pool[i] = p[np.cumsum(blen[p]) <= group]
    rows = [pool[i] for i in rng.integers(0, len(pool), size=M)]
    rpt = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    col = np.concatenate(rows).astype(np.int32)
    val = lambda n: rng.uniform(-1, 1, n) * rng.choice([1.0, 2.0 ** 30, 2.0 ** -30, 0.0], n)
    return (rpt, col, val(len(col)), K), (brpt, bcol, val(len(bcol)), N)


# a workgroup takes 16 rows per pass; one pass up to 8,192 rows, two up to
# 16,384, else four
@pytest.mark.parametrize("M", [1, 15, 17, 8192, 8193, 16384, 16385, 20000])
@pytest.mark.parametrize("group,N", [(32, 97), (32, (1 << 27) - 1), (32, 1 << 27), (64, 97), (64, (1 << 26) - 1), (64, (1 << 31) - 1)])
def test_short_rows(gpu, M, group, N):
    bm = gpu
    rng = np.random.default_rng(M * 131 + group + N % 1009)
    A, B = _operands(rng, M, N, group)
    R = oracle.brmerge_precise(A, B, nthreads=4)
    Ah, Bh = csr_from_tuple(A), csr_from_tuple(B)
    old = bm.get_param("small_fused")
    try:
        for fused in (1, 0):
            bm.set_param("small_fused", fused)
            assert_csr_equal(bm.brmerge_precise(Ah, Bh), R)
            assert_csr_equal(bm.brmerge_upper(Ah, Bh), R)
    finally:
        bm.set_param("small_fused", old)
