"""Prep of few rows and columns over a long k: the norms in one launch, the residues and the ordered
sums in a second.  Same chains in the same order as the single launch, so every output bit and counter
equals the single launch's (forced with oz2_debug_force_prep_split) and the oracle's: row counts on the
edges of the norms' 16-row workgroups and the 32-row blocks, columns on those of the 4-column workgroups
and 8-column blocks, k around the pipelined groups (32 x 8 and 16 x 8 for rows, 4 x 128 for columns) and
the 128-deep tiles, two- and three-word digits, rows and columns with NaN / Inf, zero ones, and ones that
need the rescaled norms; the other digit layout, handles without summaries, plan replays and shared
operands (no reconstruct descriptors beside the norms)."""
import ctypes as C

import numpy as np
import pytest

import ggemm as G
import oracle_lib as O
from gpu_util import dev, same_bits, say
from test_gpu_grouped import Case, kernel_handle, run
from test_gpu_reuse import Workload

pytestmark = pytest.mark.gpu

SHAPES = {   # at least 2^24 elements of A and B each, in few blocks
    "edges": [(33, 17, 130000), (8, 3, 129999), (41, 34, 65537), (1, 40, 98305)],
    "groups": [(49, 9, 130000), (48, 8, 70000), (15, 4, 130001), (16, 5, 129000), (17, 3, 90000), (47, 1, 100001)],
    "short_tail": [(64, 80, 120001), (65, 2, 127 * 1024), (7, 9, 40)],
}


def special(case):
    h = case.hp[0]
    h.A[5 + 7 * h.lda] = np.nan
    h.A[9 + 100 * h.lda] = np.inf
    h.A[3:3 + h.lda * h.k:h.lda] = 0.0
    h.A[32:32 + h.lda * h.k:h.lda] *= 1e200
    h.B[11 + 2 * h.ldb] = -np.inf
    h.B[2 * h.ldb + 4000:2 * h.ldb + 4020] = np.inf     # more infinities than a summary lists
    h.B[5 * h.ldb:6 * h.ldb] *= 1e-200
    h.B[6 * h.ldb:7 * h.ldb] = 0.0
    case.alloc()


@pytest.mark.parametrize("N", [0, 18])
@pytest.mark.parametrize("name", sorted(SHAPES))
def test_two_pass_prep(name, N):
    say(f"two-pass prep: {name}, N {N}")
    case = Case(SHAPES[name], 77, phi=1.0, beta=0.5)
    special(case)
    cfg = G.Config(N, 1e-15, 1, G.REPAIR_COUNT)
    outs, stats = [], []
    for force in (0, 1):
        G.lib().oz2_debug_force_prep_split(force)
        try:
            rc, st = run(case, G.PATH_EMU_GROUPED, cfg, min_k=32)
        finally:
            G.lib().oz2_debug_force_prep_split(0)
        assert rc == 0
        outs.append([case.C(g).copy() for g in range(len(case.hp))])
        stats.append((st.num_uncertified, st.num_safety_fallback, st.moduli_min, st.moduli_max))
        assert st.kernel_launches == (7 if force == 0 else 6)
    assert stats[0] == stats[1]
    for a, b in zip(*outs):
        assert same_bits(a, b)
    g = 1 if name == "short_tail" else 2   # against the oracle: a problem without special rows
    h = case.hp[g]
    n_mod = N or O.oracle().oz2o_choose_num_moduli(h.k, 1e-15)
    ref, _ = h.emulate(O.REPAIR_COUNT, n_mod)
    assert same_bits(outs[0][g], ref)


@pytest.mark.parametrize("env", [{"GGEMM_DIGITS_COLMAJOR": "1"}, {"GGEMM_SAFETY_CHAINS": "1"}])
def test_two_pass_handles(env):
    say(f"two-pass prep: {env}")
    case = Case(SHAPES["edges"], 78, phi=1.0, beta=0.5)
    special(case)
    outs = []
    for force in (0, 1):
        G.lib().oz2_debug_force_prep_split(force)
        try:
            with kernel_handle(case, None, **env) as hd:
                rc, st = run(case, G.PATH_EMU_GROUPED, G.Config(0, 1e-15, 1, G.REPAIR_ON), handle=hd)
        finally:
            G.lib().oz2_debug_force_prep_split(0)
        assert rc == 0
        outs.append(([case.C(g).copy() for g in range(len(case.hp))], st.num_repaired, st.num_safety_fallback,
                     st.kernel_launches + force))
    assert outs[0][1:] == outs[1][1:]
    for a, b in zip(outs[0][0], outs[1][0]):
        assert same_bits(a, b)


def test_two_pass_plan_replays():
    """A plan of the two launches replayed on data with NaN / Inf rows and columns and on finite data in
    turn, against the single launch's direct calls."""
    shapes = SHAPES["edges"]
    X, Y = Case(shapes, 79, phi=1.0, beta=0.5), Case(shapes, 80, phi=1.0, beta=0.5)
    special(X)
    cfg = G.Config(0, 1e-15, 1, G.REPAIR_ON)
    want = []
    G.lib().oz2_debug_force_prep_split(1)
    try:
        for case in (X, Y):
            rc, st = run(case, G.PATH_EMU_GROUPED, cfg)
            assert rc == 0 and st.kernel_launches == 6
            want.append([case.C(g).copy() for g in range(len(shapes))])
    finally:
        G.lib().oz2_debug_force_prep_split(0)
    h = G.Handle(len(shapes), *X.sizes())
    err = C.c_int(0)
    plan = G.lib().ggemm_make_plan_ex(h.h, G.PATH_EMU_GROUPED, C.byref(cfg), G.problems_array(X.problems()), len(shapes),
                                      C.byref(err))
    assert plan, err.value
    try:
        st = G.Stats()
        assert G.lib().ggemm_plan_get_stats(plan, C.byref(st)) == 0 and st.kernel_launches == 7
        ptr = lambda ts: (C.c_void_p * len(shapes))(*[t.data_ptr() for t in ts])  # noqa: E731
        for rep, case in enumerate((X, Y, Y, X)):
            say(f"two-pass plan replay {rep}")
            case.reset_C()
            assert G.lib().ggemm_plan_update_pointers(plan, ptr(case.dA), ptr(case.dB), ptr(case.dC)) == 0
            assert G.lib().ggemm_execute_plan(plan, None) == 0
            for g, w in enumerate(want[0 if case is X else 1]):
                assert same_bits(case.C(g), w), (rep, g)
    finally:
        G.lib().ggemm_destroy_plan(plan)
        h.close()


@pytest.mark.parametrize("share", ["A", "B"])
def test_two_pass_shared_operand(share):
    say(f"two-pass prep: shared {share}")
    m, n, k = (60, 41, 130000) if share == "A" else (41, 60, 130000)
    w = Workload("shared", 3, m, n, k, share == "A", share == "B", 1 if share == "A" else 3, 3 if share == "A" else 1, 7)
    w.hA[0][3 + 5 * m] = np.nan
    w.hA[-1][4 + 700 * m] = np.inf
    w.hB[0][9 + 2 * k] = -np.inf
    w.dA, w.dB = [dev(a) for a in w.hA], [dev(b) for b in w.hB]
    cfg = G.Config(0, 1e-15, 1, G.REPAIR_COUNT)
    with G.Handle(w.G, *w.sizes()) as h:
        rr, sr, cr = w.run(h, G.PATH_EMU_GROUPED_REUSE, cfg)
        G.lib().oz2_debug_force_prep_split(1)
        try:
            rb, sb, cb = w.run(h, G.PATH_EMU_GROUPED, cfg)
        finally:
            G.lib().oz2_debug_force_prep_split(0)
    assert rr == rb == 0
    assert (sr.reuse_enabled, sr.num_unique_A, sr.num_unique_B) == (1, *w.expect)
    assert (sr.kernel_launches, sb.kernel_launches) == (7, 6)
    assert (sr.num_uncertified, sr.num_safety_fallback) == (sb.num_uncertified, sb.num_safety_fallback)
    for g in range(w.G):
        assert same_bits(cr[g], cb[g]), g
