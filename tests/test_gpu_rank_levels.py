"""GPU parity of the register tier's bitmap ranks (rmed.hip) against the
oracle, bit for bit: rows whose column span sits on both sides of every edge
where the top level's shift changes (a level holds 64 columns per word, 256
words for rows of up to 256 products and one per product above, and every
level below spans 64 times as much), up to 2^31 - 1 columns; rows of distinct
columns, of columns met at most twice, and of columns met by many lists."""
import numpy as np
import pytest

import oracle
from tests._util import assert_csr_equal, csr_from_tuple

pytestmark = pytest.mark.gpu


def _rows(rng, ips, spans, N, shape):
    """A and B for rows of the given product counts: row i's columns lie in a
    window of spans[i] columns and include both ends of it.  shape: every
    column in one list ("distinct"), in at most two ("pairs"), or in up to 64
    ("deep")."""
    arpt, brpt, bcol = [0], [0], []
    for ip, span in zip(ips, spans):
        span = min(span, N)
        L = int(rng.integers(40, 65))
        c0 = int(rng.integers(0, N - span + 1))
        ends = np.array([0, span - 1])
        if shape == "distinct":
            n = min(ip, span)
            cols = np.unique(np.concatenate([ends, rng.choice(span, n, replace=False) if span < 1 << 22
                                             else rng.integers(0, span, n)]))[:ip]
            cols[-1] = span - 1
            where = rng.integers(0, L, len(cols))
        elif shape == "pairs":
            cols = np.unique(np.concatenate([ends, rng.integers(0, span, ip // 2)]))[:ip // 2]
            cols[-1] = span - 1
            first = rng.integers(0, L, len(cols))
            cols, where = np.concatenate([cols, cols]), np.concatenate([first, (first + 1) % L])
        else:
            pool = np.unique(np.concatenate([ends, rng.integers(0, span, max(2, ip // 20))]))
            cols, where = [], []
            for l in range(L):
                c = rng.choice(pool, min(len(pool), max(1, ip // L)), replace=False)
                cols.append(c)
                where.append(np.full(len(c), l))
            cols, where = np.concatenate(cols), np.concatenate(where)
        for l in range(L):
            c = np.sort(cols[where == l])
            bcol.append(c + c0)
            brpt.append(brpt[-1] + len(c))
        arpt.append(arpt[-1] + L)
    K = len(brpt) - 1
    bcol = np.concatenate(bcol).astype(np.int32)
    val = lambda n: rng.uniform(-1, 1, n) * rng.choice([1.0, 2.0 ** 30, 2.0 ** -30], n)  # noqa: E731
    A = (np.array(arpt, np.int32), np.arange(K, dtype=np.int32), val(K), K)
    B = (np.array(brpt, np.int32), bcol, val(len(bcol)), N)
    return A, B


@pytest.mark.parametrize("shape", ["distinct", "pairs", "deep"])
@pytest.mark.parametrize("ncols", [1 << 16, (1 << 16) + 1, 1 << 20, 1 << 26, (1 << 31) - 1])
@pytest.mark.parametrize("cap", [256, 512, 1024, 2048])
def test_rank_level_edges(gpu, cap, ncols, shape):
    bm = gpu
    rng = np.random.default_rng(cap * 31 + ncols % 1009 + len(shape))
    words = max(256, cap)
    spans = []
    for sh in (0, 6, 12):
        edge = (64 * words) << sh
        spans += [edge - 1, edge, edge + 1, edge + (64 << sh)]
    spans += [70, 4096, 1 << 30]
    spans = [max(64, min(s, ncols)) for s in spans]
    ips = [int(x) for x in rng.integers(cap // 2 + 1, cap + 1, len(spans))]
    if shape == "distinct":
        ips = [min(i, s) for i, s in zip(ips, spans)]
    A, B = _rows(rng, ips, spans, ncols, shape)
    R = oracle.brmerge_precise(A, B, nthreads=4)
    Ah, Bh = csr_from_tuple(A), csr_from_tuple(B)
    old = bm.get_param("wmed_cap")
    bm.set_param("wmed_cap", cap)
    try:
        for f in (bm.brmerge_precise, bm.brmerge_upper):
            assert_csr_equal(f(Ah, Bh), R)
    finally:
        bm.set_param("wmed_cap", old)


@pytest.mark.parametrize("dmin,dmax", [(9, 14), (17, 22)], ids=["to_256", "to_512"])
@pytest.mark.parametrize("rows", [16383, 32769, 140011])
def test_several_rows_per_wavefront(gpu, rows, dmin, dmax):
    """Row lists long enough for one, two and eight rows per wavefront (and
    last wavefronts and shares of the XCDs that are not full), banded rows with
    empty lists among them."""
    bm = gpu
    rng = np.random.default_rng(rows + dmin)

    def banded(lo, hi, empty):
        deg = rng.integers(lo, hi + 1, rows)
        deg[rng.random(rows) < empty] = 0
        r = np.repeat(np.arange(rows), deg)
        key = np.unique(r * rows + np.clip(r + rng.integers(-40, 41, len(r)), 0, rows - 1))
        rpt = np.concatenate([[0], np.cumsum(np.bincount(key // rows, minlength=rows))]).astype(np.int32)
        return rpt, (key % rows).astype(np.int32), rng.uniform(-1, 1, len(key)), rows

    A, B = banded(dmin, dmax, 0.0), banded(dmin, dmax, 0.1)
    R = oracle.brmerge_precise(A, B, nthreads=8)
    Ah, Bh = csr_from_tuple(A), csr_from_tuple(B)
    for f in (bm.brmerge_precise, bm.brmerge_upper):
        assert_csr_equal(f(Ah, Bh), R)
