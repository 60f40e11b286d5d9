"""Who finishes a product of short rows, by the kernels that ran: the fused
kernel in one launch (two where a row is too long for groups of 32 lanes), and
the general pipeline where the fused kernel's scan is given up (small_looks 0:
at the first look without news, every kernel ends as ever), without a second try in groups of 64.
C is the oracle's either way, and operands out of order are refused."""
import numpy as np
import pytest

import oracle
from tests._util import assert_csr_equal, csr_from_tuple

pytestmark = pytest.mark.gpu


def _operands(rng, M, per, longest=None):
    K, N = 4000, 700
    lens = np.full(M, per)
    lens[M // 2] = longest or per
    acol = np.concatenate([np.sort(rng.choice(K, n, replace=False)) for n in lens]).astype(np.int32)
    A = (np.concatenate([[0], np.cumsum(lens)]).astype(np.int32), acol, rng.uniform(-1, 1, len(acol)), K)
    B = (np.arange(K + 1, dtype=np.int32), rng.integers(0, N, K).astype(np.int32), rng.uniform(-1, 1, K), N)
    return A, B


def _kernels(bm, f):
    bm.set_param("profile", 1)
    bm.prof_reset()
    try:
        r = f()
        return r, {k: v[0] for k, v in bm.prof_report().items()}
    finally:
        bm.set_param("profile", 0)


@pytest.mark.parametrize("looks", [None, 0])
@pytest.mark.parametrize("M,per,longest", [(M, *p) for M in (1, 16, 17, 3000, 20000)
                                           for p in ((20, None), (20, 40), (50, None)) if M > 1 or p[1] is None])
def test_finisher(gpu, M, per, longest, looks):
    bm = gpu
    rng = np.random.default_rng(M + per + (longest or 0))
    A, B = _operands(rng, M, per, longest)
    R = oracle.brmerge_precise(A, B, nthreads=4)
    Ah, Bh = csr_from_tuple(A), csr_from_tuple(B)
    bad = csr_from_tuple(B)
    bad.col = bad.col.copy()
    bad.col[A[1][0]] = -1
    old = bm.get_param("small_looks")
    try:
        if looks is not None:
            bm.set_param("small_looks", looks)
        for f in (bm.brmerge_precise, bm.brmerge_upper):
            C, ran = _kernels(bm, lambda: f(Ah, Bh))
            assert_csr_equal(C, R)
            if looks == 0:
                # (with a few workgroups all may be done before the first look)
                assert ran["k_small"] == 1 or M < 3000, ran
                assert "k_rowstats" in ran or M < 3000, ran
            else:
                assert ran["k_small"] == (2 if longest else 1) and "k_rowstats" not in ran, ran
            with pytest.raises(bm.BrmError) as e:
                f(Ah, bad)
            assert e.value.status == 1
    finally:
        bm.set_param("small_looks", old)


def test_looks_range(gpu):
    bm = gpu
    old = bm.get_param("small_looks")
    for v in (-1, (1 << 20) + 1):
        with pytest.raises(bm.BrmError):
            bm.set_param("small_looks", v)
    assert bm.get_param("small_looks") == old
