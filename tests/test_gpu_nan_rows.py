"""Rows of A and columns of B that hold a NaN are read no further by prep's norm pass: NaNs in the first
pipelined group, in a later one, in the last partial group and in the last element, with infinities
before and after them, next to rows with infinities only and finite ones; bitwise against the oracle
with equal counters in the three repair modes."""
import numpy as np
import pytest

import ggemm as G
import oracle_lib as O
from gpu_util import say
from test_gpu_grouped import Case, check_case, kernel_handle, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [255, 1024, 1500, 2561])
@pytest.mark.parametrize("repair,mode", [(G.REPAIR_OFF, O.REPAIR_OFF), (G.REPAIR_COUNT, O.REPAIR_COUNT),
                                         (G.REPAIR_ON, O.REPAIR_ON)])
def test_nan_rows(k, repair, mode):
    say(f"NaN rows, k {k}, repair {repair}")
    case = Case([(45, 21, k), (33, 9, k // 2)], 17, phi=1.5, beta=0.5)
    for h in case.hp:
        a, b, K = h.lda, h.ldb, h.k
        for i, at in ((0, 3), (1, K // 2), (2, K - 1), (3, K - 9), (40 % h.m, 0)):
            h.A[i + at * a] = np.nan
        h.A[0 + (K - 2) * a] = np.inf      # past the row's NaN
        h.A[2 + 1 * a] = -np.inf           # before it
        h.A[5 + (K - 1) * a] = np.inf      # no NaN in the row
        h.A[5 + 7 * a] = -np.inf
        for j, at in ((0, 0), (1, K // 2), (2, K - 1)):
            h.B[at + j * b] = np.nan
        h.B[(K - 1) + 0 * b] = np.inf
        h.B[5 + 3 * b] = np.inf
    case.alloc()
    cfg = G.Config(0, 1e-15, 1, repair)
    with kernel_handle(case, None, GGEMM_STATS_REPAIR="1") as hd:
        rc, st = run(case, G.PATH_EMU_GROUPED, cfg, handle=hd)
    assert rc == 0
    check_case(case, G.PATH_EMU_GROUPED, cfg, st, mode)


@pytest.mark.parametrize("k", [255, 1500, 4200])
@pytest.mark.parametrize("scale_a,scale_b", [(1e280, 1e-300), (1e-290, 1e250)])
def test_nan_rows_of_extreme_magnitude(k, scale_a, scale_b):
    """Magnitudes whose squares need the rescaled second read of a row, in rows and columns that hold a
    NaN, infinities, both in either order, or neither."""
    say(f"NaN rows of extreme magnitude, k {k}")
    case = Case([(45, 21, k), (33, 9, k)], 18, phi=1.0, beta=0.5)
    for h in case.hp:
        h.A *= scale_a
        h.B *= scale_b
        a, b, K = h.lda, h.ldb, h.k
        h.A[0 + 3 * a], h.A[0 + (K - 2) * a] = np.nan, np.inf
        h.A[1 + 3 * a], h.A[1 + (K - 2) * a] = -np.inf, np.nan
        h.A[2 + (K // 2) * a] = np.nan
        h.A[4 + (K // 2) * a] = np.inf
        h.B[0], h.B[K - 1] = np.nan, np.inf
        h.B[b], h.B[b + K - 1] = np.inf, np.nan
        h.B[2 * b + K // 2] = np.nan
        h.B[5 * b + K // 2] = -np.inf
    case.alloc()
    cfg = G.Config(0, 1e-15, 1, G.REPAIR_ON)
    with kernel_handle(case, None, GGEMM_STATS_REPAIR="1") as hd:
        rc, st = run(case, G.PATH_EMU_GROUPED, cfg, handle=hd)
    assert rc == 0
    check_case(case, G.PATH_EMU_GROUPED, cfg, st, O.REPAIR_ON)
