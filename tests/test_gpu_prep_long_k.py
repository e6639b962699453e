"""Prep of few rows and columns over a long k: the norms in one launch, the residues and the ordered
sums in a second.  Same chains in the same order as the single launch, so every output bit and counter
equals the single launch's (forced with oz2_debug_force_prep_split) and the oracle's: row counts on the
edges of the 8-row waves and 32-row blocks, columns on those of the 2-column waves, k around the
pipelined groups (32 x 8 and 8 x 128) and the 128-deep tiles, two- and three-word digits, rows and
columns with NaN / Inf, zero ones, and ones that need the rescaled norms."""
import numpy as np
import pytest

import ggemm as G
import oracle_lib as O
from gpu_util import same_bits, say
from test_gpu_grouped import Case, run

pytestmark = pytest.mark.gpu

SHAPES = {   # at least 2^24 elements of A and B each, in few blocks
    "edges": [(33, 17, 130000), (8, 3, 129999), (41, 34, 65537), (1, 40, 98305)],
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
    g = 2 if name == "edges" else 1   # against the oracle: a problem without special rows
    h = case.hp[g]
    n_mod = N or O.oracle().oz2o_choose_num_moduli(h.k, 1e-15)
    ref, _ = h.emulate(O.REPAIR_COUNT, n_mod)
    assert same_bits(outs[0][g], ref)
