"""Rows of B that are out of order, used by rows that the fused short-row path
merges (beside its check of B): a column twice, next to each other or apart,
in one row or in every row, and columns past N that meet a column of the row
once shifted into the packed sort keys.  Each is refused with status 1 by
every entry, in groups of 32 and of 64 lanes and on both sides of the widths
where the packed keys end, and a product in order after it is right."""
import numpy as np
import pytest

import oracle
from tests._util import assert_csr_equal, csr_from_tuple

pytestmark = pytest.mark.gpu


def _operands(rng, group, N):
    """1,000 rows of `per` lists with `per` entries each (at most `group`
    products), B's rows from a pool of 40 columns."""
    per, K = (5, 300) if group == 32 else (8, 300)
    pool = np.sort(rng.choice(N - 1, 40, replace=False))
    pool[-1] = N - 1
    bcol = np.concatenate([np.sort(rng.choice(pool, per, replace=False)) for _ in range(K)]).astype(np.int32)
    acol = np.concatenate([np.sort(rng.choice(K, per, replace=False)) for _ in range(1000)]).astype(np.int32)
    A = (np.arange(1001, dtype=np.int32) * per, acol, rng.uniform(-1, 1, len(acol)), K)
    B = (np.arange(K + 1, dtype=np.int32) * per, bcol, rng.uniform(-1, 1, len(bcol)), N)
    return A, B, per


def _spoil(B, per, group, N, how):
    col = B[1].copy().reshape(-1, per)
    rows = slice(None) if how == "all" else slice(17, 18)
    if how == "apart":
        col[rows, per - 1] = col[rows, 0]
    elif how == "past":
        col[rows, per - 1] = col[rows, 0].astype(np.int64) + (1 << (27 if group == 32 else 26))
    else:
        col[rows, 1] = col[rows, 0]
    return (B[0], col.reshape(-1), B[2], N)


@pytest.mark.parametrize("how", ["one", "all", "apart", "past"])
@pytest.mark.parametrize("group,N", [(32, 97), (32, (1 << 27) - 1), (32, 1 << 27), (64, 97), (64, (1 << 26) - 1),
                                     (64, 1 << 26)])
def test_refused(gpu, group, N, how):
    bm = gpu
    rng = np.random.default_rng(group + N % 1009 + len(how))
    A, B, per = _operands(rng, group, N)
    R = oracle.brmerge_precise(A, B, nthreads=4)
    Ah, Bh, bad = csr_from_tuple(A), csr_from_tuple(B), csr_from_tuple(_spoil(B, per, group, N, how))
    dev = [bm.DeviceCSR.upload(x) for x in (Ah, Bh, bad)]
    try:
        for f in (bm.brmerge_precise, bm.brmerge_upper):
            with pytest.raises(bm.BrmError) as e:
                f(Ah, bad)
            assert e.value.status == 1
            assert_csr_equal(f(Ah, Bh), R)
        for upper in (False, True):
            with pytest.raises(bm.BrmError) as e:
                bm.spgemm_dev(dev[0], dev[2], upper=upper)
            assert e.value.status == 1
            C = bm.spgemm_dev(dev[0], dev[1], upper=upper)
            assert_csr_equal(C.download(), R)
            C.free()
    finally:
        for d in dev:
            d.free()
