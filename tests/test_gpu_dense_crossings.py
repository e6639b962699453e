"""The dot pass defers a tile's dense crossings to the crossings pass whatever their number: tiles with
just under, at and past the compact form's 256 crossings, all uncertified entries repaired, bitwise
against the oracle with equal counters, and equal to the handle that defers nothing."""
import numpy as np
import pytest

import ggemm as G
import oracle_lib as O
from gpu_util import same_bits, say
from test_gpu_grouped import Case, check_case, kernel_handle, run

pytestmark = pytest.mark.gpu

CFG = G.Config(0, 1e-15, 1, G.REPAIR_ON)


@pytest.mark.parametrize("rows,cols", [(16, 16), (17, 16), (24, 30), (31, 32)])
@pytest.mark.parametrize("beta", [0.0, 0.5])
def test_dense_crossings(rows, cols, beta):
    say(f"dense crossings {rows} x {cols} per tile, beta {beta}")
    outs = []
    for form in ("", "tile"):
        case = Case([(130, 128, 300), (64, 64, 257)], 91, phi=4.0, beta=beta)
        rng = np.random.default_rng(3)
        for h in case.hp:   # all but `rows` rows and `cols` columns of each 64 x 64 tile hold a NaN
            for r0 in range(0, h.m, 64):
                for i in rng.permutation(np.arange(r0, min(r0 + 64, h.m)))[rows:]:
                    h.A[i + 7 * h.lda] = np.nan
            for c0 in range(0, h.n, 64):
                for j in rng.permutation(np.arange(c0, min(c0 + 64, h.n)))[cols:]:
                    h.B[5 + j * h.ldb] = np.nan
        case.alloc()
        env = {"GGEMM_DOT_FORM": form} if form else {}
        with kernel_handle(case, None, GGEMM_STATS_REPAIR="1", **env) as hd:
            rc, st = run(case, G.PATH_EMU_GROUPED, CFG, handle=hd)
        assert rc == 0
        check_case(case, G.PATH_EMU_GROUPED, CFG, st, O.REPAIR_ON)
        assert st.num_repaired >= 0.5 * rows * cols
        outs.append([case.C(g).copy() for g in range(2)])
    for a, b in zip(*outs):
        assert same_bits(a, b)


@pytest.mark.parametrize("bad", ["rows", "all", "half"])
@pytest.mark.parametrize("shape", [(88, 80, 300), (80, 121, 257), (64, 17, 129), (17, 16, 300), (16, 57, 300), (11, 24, 129), (80, 57, 64)])
def test_dense_edge_tiles(shape, bad):
    """Tiles over the problem's edge whose entries all (or half of them) take their chains -- rows and
    columns with an infinity, no summaries: bitwise against the oracle with equal counters, and equal to
    the handle that defers nothing."""
    say(f"dense edge tiles {shape}, {bad}")
    outs = []
    for form in ("", "tile", "blocks"):
        case = Case([shape], 23, phi=1.0, beta=0.5)
        h = case.hp[0]
        for i in range(0, h.m, 2 if bad == "half" else 1):
            h.A[i + (3 * i % h.k) * h.lda] = np.inf if i % 3 else -np.inf
        if bad == "all":
            for j in range(h.n):
                h.B[(5 * j) % h.k + j * h.ldb] = np.inf if j % 2 else np.nan
        case.alloc()
        env = {"GGEMM_DOT_FORM": form} if form else {}
        with kernel_handle(case, None, GGEMM_STATS_REPAIR="1", GGEMM_SAFETY_CHAINS="1", **env) as hd:
            rc, st = run(case, G.PATH_EMU_GROUPED, CFG, handle=hd)
        assert rc == 0
        check_case(case, G.PATH_EMU_GROUPED, CFG, st, O.REPAIR_ON)
        assert st.num_safety_fallback >= h.m * h.n // 2
        outs.append(case.C(0).copy())
    assert same_bits(outs[0], outs[1]) and same_bits(outs[0], outs[2])


@pytest.mark.parametrize("rows,cols", [(3, 4), (5, 0), (0, 6), (12, 9), (1, 1), (7, 40)])
def test_flagged_lines(rows, cols):
    """Whole rows and columns of every 64 x 64 tile take their chains (infinities, no summaries), with some
    tiles free of either: deferred lines, mixed tiles in the dense form, edge tiles; bitwise against the
    oracle with equal counters, and equal to the handles that defer nothing / run block by block."""
    say(f"flagged lines: {rows} rows, {cols} columns per tile")
    outs = []
    for form in ("", "tile", "blocks"):
        case = Case([(150, 200, 300), (64, 128, 65)], 29, phi=1.0, beta=0.5)
        rng = np.random.default_rng(5)
        for h in case.hp:
            for r0 in range(0, h.m, 64):
                for i in rng.permutation(np.arange(r0, min(r0 + 64, h.m)))[:0 if r0 == 64 else rows]:
                    h.A[i + (7 * i % h.k) * h.lda] = np.inf
            for c0 in range(0, h.n, 64):
                for j in rng.permutation(np.arange(c0, min(c0 + 64, h.n)))[:0 if c0 == 64 else cols]:
                    h.B[5 * j % h.k + j * h.ldb] = -np.inf if j % 2 else np.nan
        case.alloc()
        env = {"GGEMM_DOT_FORM": form} if form else {}
        with kernel_handle(case, None, GGEMM_STATS_REPAIR="1", GGEMM_SAFETY_CHAINS="1", **env) as hd:
            rc, st = run(case, G.PATH_EMU_GROUPED, CFG, handle=hd)
        assert rc == 0
        check_case(case, G.PATH_EMU_GROUPED, CFG, st, O.REPAIR_ON)
        outs.append([case.C(g).copy() for g in range(2)])
    for a, b, c in zip(*outs):
        assert same_bits(a, b) and same_bits(a, c)
