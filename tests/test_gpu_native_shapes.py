"""The native FP64 GEMM's tile shapes on the edges of tiles, of the 16-, 64- and 128-deep k stages and of
the rule that chooses: 32 x 32 tiles (few outputs), 16 x 128 and 32 x 128 tiles (many thin problems),
128 x 128 tiles (filled rounds); each group's shape is the one it is meant for.  Every shape takes the same k-ordered chain per entry, so each result
equals the 64 x 64 kernel's (forced with GGEMM_F64_TILE) bit for bit; that kernel is held to the
componentwise gamma_n bound against the host's extended-precision dots."""
import numpy as np
import pytest

import ggemm as G
from gpu_util import same_bits, say
from test_f64_schedule import CHAIN, SHORT, T16, T32, T128, schedule
from test_gpu_grouped import Case, kernel_handle, run

pytestmark = pytest.mark.gpu

CFG = G.Config(0, 1e-15, 1, G.REPAIR_ON)
EDGES = [(32, 32, 128), (33, 31, 127), (31, 33, 129), (64, 1, 255), (1, 64, 256), (70, 50, 257), (1, 1, 1), (40, 40, 0),
         (0, 5, 5), (48, 48, 385), (20, 20, 63), (20, 20, 64), (20, 20, 65), (20, 20, 193)]
GROUPS = {   # name: tile shape, problems
    # few outputs, 32 x 32 tiles: 64-deep stages up to k = 512, 128-deep ones with a longer k in the group
    "short_edges": (SHORT, EDGES),
    "chain_edges": (CHAIN, EDGES + [(32, 33, 513)]),   # one to five stages, k = 0
    "chain_long_k": (CHAIN, [(70, 50, 9000), (65, 1, 8191), (5, 40, 12345)]),
    "short_512": (SHORT, [(64, 60, 511), (31, 32, 512), (33, 1, 448)]),
    "chain_513": (CHAIN, [(64, 60, 513), (31, 32, 512), (33, 1, 640)]),
    "chain_256_tiles": (CHAIN, [(32 * 15, 32 * 17, 700), (20, 20, 650)]),
    "chain_257_tiles": (SHORT, [(32 * 16, 32 * 16, 700), (20, 20, 650)]),   # 64-deep ones past 256 tiles
    "short_alpha0": (SHORT, [(50, 40, 300, 0.0, 0.5), (50, 40, 300, -1.0, 0.0)]),
    # enough thin problems for the thin tiles
    "thin16": (T16, [(1 + i % 16, 120 + i % 20, 1 + i % 50) for i in range(300)]),
    "thin32": (T32, [(1 + i % 32, 250 + i % 9, 15 + i % 35) for i in range(300)]),
    # one full round of 128 x 128 tiles (two per compute unit) and no edges
    "tile128": (T128, [(4096, 2048, 40)]),
}


@pytest.mark.parametrize("beta", [0.0, -0.5])
@pytest.mark.parametrize("name", sorted(GROUPS))
def test_native_shapes(name, beta):
    say(f"native shapes: {name}, beta {beta}")
    shape, group = GROUPS[name]
    assert schedule(group)[:2] == (0, shape)
    outs = []
    for env in ({}, {"GGEMM_F64_TILE": "64"}):
        case = Case(group, 41, phi=1.0, alpha=1.5, beta=beta)
        with kernel_handle(case, None, **env) as hd:
            rc, st = run(case, G.PATH_NATIVE_GROUPED, CFG, handle=hd)
        assert rc == 0 and st.kernel_launches == 1
        outs.append([case.C(g).copy() for g in range(len(case.hp))])
    for g, (a, b) in enumerate(zip(*outs)):
        assert same_bits(a, b), (g, group[g])
    for g, h in enumerate(case.hp):
        if h.m == 0 or h.n == 0 or h.m * h.n * h.k > 10 ** 8:
            continue
        h.reference()
        gate, _ = h.gate(outs[0][g])
        assert gate <= 1.0, (g, gate)


UNDERFLOW = {   # every product underflows to -0: the sign of the result tells how far the chain is padded
    "short": [(20, 20, k) for k in (1, 4, 8, 12, 15, 16, 20, 60, 64, 68, 130)],
    "chain": [(20, 20, k) for k in (4, 16, 600, 624, 1020, 1032)],
    "thin16": [(1 + i % 16, 130, 4 + i % 17) for i in range(300)],
    "thin32": [(17 + i % 16, 250, 4 + i % 17) for i in range(300)],
}


@pytest.mark.parametrize("name", sorted(UNDERFLOW))
def test_underflow_sign(name):
    say(f"underflow: {name}")
    assert schedule(UNDERFLOW[name])[1] == {"short": SHORT, "chain": CHAIN, "thin16": T16, "thin32": T32}[name]
    outs = []
    for env in ({}, {"GGEMM_F64_TILE": "64"}, {"GGEMM_F64_TILE": "128"}):
        case = Case(UNDERFLOW[name], 5)
        for h in case.hp:
            h.A[:], h.B[:] = 1e-200, -1e-200
        case.alloc()
        with kernel_handle(case, None, **env) as hd:
            rc, _ = run(case, G.PATH_NATIVE_GROUPED, CFG, handle=hd)
        assert rc == 0
        outs.append([case.C(g).copy() for g in range(len(case.hp))])
    for g, h in enumerate(case.hp):
        assert np.array_equal(outs[1][g], np.zeros(h.m * h.n))
        assert np.signbit(outs[1][g]).all() == (h.k % 16 == 0)   # +0 once the chain is padded past k
        assert same_bits(outs[0][g], outs[1][g]) and same_bits(outs[2][g], outs[1][g]), (g, UNDERFLOW[name][g])
