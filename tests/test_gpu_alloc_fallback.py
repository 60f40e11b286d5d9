"""Device memory that runs out while a product of long rows is set up: every
allocation of the call fails in turn, in one wave of rows and in several that
overlap.  The product is right or out of memory, and with the column tiles'
tables it is out of memory at no more allocations than without: where a table
does not fit, the engine without tables runs."""
import numpy as np
import pytest

import oracle
from tests._util import as_tuple, assert_csr_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("upper", [False, True])
@pytest.mark.parametrize("ws", [0, 1 << 19])
def test_every_allocation(gpu, ws, upper):
    bm = gpu
    L = bm.lib()
    A = bm.gen.rmat(11, seed=3)
    R = oracle.brmerge_precise(as_tuple(A), as_tuple(A), nthreads=4)
    f = bm.brmerge_upper if upper else bm.brmerge_precise
    names = ("force_long", "long_tiles", "ws_budget_bytes")
    saved = {k: bm.get_param(k) for k in names}
    refused, ran = {}, {}
    try:
        bm.set_param("force_long", 1)
        bm.set_param("ws_budget_bytes", ws)
        for tiles in (0, 64):
            bm.set_param("long_tiles", tiles)
            refused[tiles], ran[tiles] = [], []
            for n in range(120):
                L.brm_debug_fail_alloc_after(n)
                try:
                    C = f(A, A)
                except bm.BrmError as e:
                    assert e.status == 2
                    refused[tiles].append(n)
                else:
                    assert_csr_equal(C, R)
                    ran[tiles].append(n)
                L.brm_debug_fail_alloc_after(-1)
            assert ran[tiles][-20:] == list(range(100, 120))
            waves = bm.last_stats()["long_waves"]
            assert waves == 1 if ws == 0 else waves > 1
    finally:
        L.brm_debug_fail_alloc_after(-1)
        for k, v in saved.items():
            bm.set_param(k, v)
    assert len(refused[64]) == len(refused[0]), (refused, ran)
