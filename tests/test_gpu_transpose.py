"""The device transpose against the host transpose at every number of lanes
per row (averages at and around 2, 8 and 32 entries), with empty rows, a row
of all columns, columns without entries at both ends, and no entries."""
import numpy as np
import pytest

from tests._util import assert_csr_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,lens", [
    (1, 1, (1, 1)), (257, 70000, (0, 3)), (1023, 40, (2, 2)), (1000, 500, (0, 6)), (999, 333, (8, 8)),
    (700, 90000, (9, 9)), (513, 1200, (20, 44)), (300, 4000, (33, 33)), (64, 5000, (0, 400)), (50, 60, (0, 0)),
])
def test_transpose(gpu, M, N, lens):
    bm = gpu
    rng = np.random.default_rng(M + N)
    rows = [np.sort(rng.choice(max(N - 2, 1), size=min(int(rng.integers(lens[0], lens[1] + 1)), N), replace=False)) + (N > 2)
            for _ in range(M)]
    if M > 60:
        rows[M // 2] = np.arange(min(N, 3000))  # a long row among short ones
        rows[M // 3] = np.arange(0)
    rpt = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    col = np.concatenate(rows).astype(np.int32)
    A = bm.CSR(rpt, col, rng.uniform(-1, 1, len(col)), M, N)
    dA = bm.DeviceCSR.upload(A)
    dT = dA.transpose()
    H = dT.download()
    assert (H.M, H.N) == (N, M)
    assert_csr_equal(H, A.transpose())
    dA.free()
    dT.free()
