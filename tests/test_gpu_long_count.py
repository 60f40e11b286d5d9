"""The long rows' symbolic count (k_sym_bitmap) against numpy at bitmap sizes
around its steps of 1,024 columns, around two workgroups per CU, and around
one and two passes of 2^20 columns; first and last columns always present."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1, 31, 1023, 1024, 1025, 300000, (1 << 20) - 1, 1 << 20, (1 << 20) + 1, (1 << 21) + 5])
def test_counts(gpu, N):
    bm = gpu
    rng = np.random.default_rng(N)
    K = 150
    B = [np.unique(np.concatenate([[0, N - 1], rng.integers(0, N, int(rng.integers(1, 200)))])) for _ in range(K)]
    A = [np.arange(K), np.sort(rng.choice(K, 70, replace=False)), np.array([3])]
    csr = lambda rr, n: bm.CSR(np.concatenate([[0], np.cumsum([len(r) for r in rr])]).astype(np.int32),
                               np.concatenate(rr).astype(np.int32), rng.uniform(-1, 1, sum(map(len, rr))), len(rr), n)
    old = bm.get_param("force_long")
    try:
        bm.set_param("force_long", 1)
        C = bm.brmerge_precise(csr(A, K), csr(B, N))
    finally:
        bm.set_param("force_long", old)
    want = [np.unique(np.concatenate([B[j] for j in r])) for r in A]
    np.testing.assert_array_equal(np.diff(np.asarray(C.rpt, np.int64)), [len(w) for w in want])
    np.testing.assert_array_equal(C.col, np.concatenate(want))
