"""The calls whose speed is measured: what programs have this library do, over the range they do it in.

A case is a dict of plain values; prepare() makes its inputs and the handle (or plan) that a program
keeps, run() is one pass through the C ABI (ctypes binding, coding-basic-hw-2_amd/ggemm).  Kinds:
  group   g equal problems m x n x k
  ragged  g problems, m and n log-uniform in [mn_lo, mn_hi], k in [k_lo, k_hi], a sixteenth with
          alpha = 0, alpha ~ U(-2, 2), beta ~ U(-1, 1)
  moe     the two grouped products of a mixture-of-experts layer (apps/moe_ffn.py): one problem per
          expert, row counts by Zipf popularity
  panels  block rows of an atom-blocked sparse matrix times a dense multi-vector (apps/block_sparse.py)
  shared  g problems with one common A (weights) and different B
Every problem of a case lives in one flat buffer per operand (column-major, 256-byte aligned
problems), and run() returns the whole C buffers.
"""
import ctypes as C
import math
import random
import sys
from pathlib import Path

import numpy as np
import torch

_PKG = Path(__file__).resolve().parents[1] / "coding-basic-hw-2_amd"
for _p in (str(_PKG), str(_PKG / "apps")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

import block_sparse  # noqa: E402
import ggemm as G  # noqa: E402
import moe_ffn  # noqa: E402

PATHS = {"native": G.PATH_NATIVE_GROUPED, "emu": G.PATH_EMU_GROUPED, "auto": G.PATH_AUTO,
         "reuse": G.PATH_EMU_GROUPED_REUSE}
REPAIR = {"default": G.REPAIR_DEFAULT, "off": G.REPAIR_OFF, "count": G.REPAIR_COUNT, "on": G.REPAIR_ON}
_BASE = {"path": "emu", "repair": "on", "moduli": 0, "phi": 0.5, "alpha": 1.0, "beta": 0.0, "bad": 0.0, "api": "call"}


def listed():
    def case(name, kind, **kw):
        return dict(_BASE, name=name, kind=kind, **kw)
    return [
        # one small product with a fixed number of moduli: launches and latency
        case("single_256", "group", g=1, m=256, n=256, k=256, moduli=14),
        # a serving loop without a handle: a few small odd-sized products per call
        case("noalloc_12", "ragged", g=12, mn_lo=40, mn_hi=150, k_lo=40, k_hi=150, shape_seed=3,
             repair="default", api="noalloc"),
        # a batch of equal mid-size products, accumulated
        case("uniform_1024", "group", g=64, m=1024, n=1024, k=1024, beta=0.5),
        # a ragged group from short k to long, odd sizes, some alpha = 0
        case("ragged_128", "ragged", g=128, mn_lo=64, mn_hi=4096, k_lo=16, k_hi=8192, shape_seed=20261203, phi=1.0),
        # the largest products, planned once and replayed on new output buffers
        case("large_plan", "group", g=2, m=8192, n=8192, k=16384, phi=0.0, api="plan"),
        # wide dynamic range with NaN / Inf entries, routed by the planner
        case("hard_auto", "group", g=16, m=2048, n=2048, k=2048, phi=4.0, bad=1e-3, path="auto", long_g=2, long_k=65536),
        # few outputs over a very long k, more moduli than usual, failures only counted
        case("long_k_wide", "group", g=2, m=600, n=384, k=40000, moduli=18, phi=1.0, repair="count"),
        # one weight matrix against many inputs, its residues prepared once
        case("shared_weights", "shared", g=16, m=1536, n=512, k=2048, path="reuse", repair="default"),
        # the native FP64 path on the same batch
        case("native_1024", "group", g=64, m=1024, n=1024, k=1024, beta=0.5, path="native"),
        # a Gram-like product: small output, very long k, routed by the planner
        case("gram_auto", "group", g=1, m=500, n=500, k=60000, path="auto"),
        # a mixture-of-experts layer, routed by the planner
        case("moe_auto", "moe", tokens=4096, experts=16, topk=2, d=1024, f=2048, path="auto", repair="default",
             shape_seed=7),
        # a thousand thin block rows (5 to 14 rows each), routed by the planner
        case("panels_auto", "panels", atoms=1024, basis="dz", cutoff=6.0, nrhs=128, path="auto", repair="default",
             shape_seed=11),
    ]


def _lu(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["group", "group", "gram", "small", "ragged", "moe", "panels", "shared"])
    c = dict(_BASE, phi=round(rng.uniform(0.0, 1.2), 3), beta=rng.choice([0.0, 0.0, 0.5, -0.75]),
             alpha=rng.choice([1.0, 1.0, -1.5]))
    mode = rng.choice([("emu", "on"), ("emu", "count"), ("auto", "default"), ("native", "default")])
    c.update(path=mode[0], repair=mode[1])
    if kind == "group":
        m, n, k = _lu(rng, 100, 5000), _lu(rng, 100, 5000), _lu(rng, 32, 12000)
        g = max(1, min(96, int(rng.uniform(0.2, 1.0) * 1.2e11 / (m * n * k)), int(1.2e8 / (m * k + n * k + m * n))))
        while m * n * k * g > 3e11:
            m, n, k = m // 2 + 1, n // 2 + 1, k // 2 + 1
        c.update(kind="group", g=g, m=m, n=n, k=k)
        extra = rng.random()
        if extra < 0.15:
            c.update(phi=4.0, bad=1e-3, path="auto", repair="on")
        elif extra < 0.35:
            c.update(moduli=rng.randint(13, 19), path="emu")
        elif extra < 0.5 and c["path"] != "native":
            c.update(api="plan")
    elif kind == "gram":
        c.update(kind="group", g=rng.randint(1, 3), m=_lu(rng, 64, 1000), n=_lu(rng, 64, 1000), k=_lu(rng, 8000, 90000))
        if c["path"] == "emu" and rng.random() < 0.5:
            c.update(moduli=rng.randint(17, 19))
    elif kind == "small":
        c.update(kind="ragged", g=rng.randint(1, 16), mn_lo=24, mn_hi=120, k_lo=24, k_hi=120, shape_seed=rng.randrange(10 ** 6))
        if c["path"] != "native" and rng.random() < 0.5:
            c.update(api="noalloc")
    elif kind == "ragged":
        c.update(kind="ragged", g=rng.randint(8, 128), mn_lo=64, mn_hi=_lu(rng, 500, 4096), k_lo=16, k_hi=_lu(rng, 500, 8192),
                 shape_seed=rng.randrange(10 ** 6))
    elif kind == "moe":
        c.update(kind="moe", tokens=_lu(rng, 300, 6000), experts=rng.randint(4, 24), topk=rng.randint(1, 3),
                 d=16 * rng.randint(16, 80), f=16 * rng.randint(32, 160), alpha=1.0, beta=0.0, shape_seed=rng.randrange(10 ** 6))
    elif kind == "panels":
        c.update(kind="panels", atoms=rng.randint(100, 1200), basis=rng.choice(["dz", "dz", "tz"]),
                 cutoff=round(rng.uniform(3.0, 6.5), 2), nrhs=rng.randint(16, 160), alpha=1.0, beta=0.0,
                 shape_seed=rng.randrange(10 ** 6))
    else:
        c.update(kind="shared", g=rng.randint(4, 24), m=_lu(rng, 200, 2500), n=_lu(rng, 100, 1200), k=_lu(rng, 200, 4000),
                 path="reuse", repair="default", alpha=1.0)
    return c


def _shapes(c):
    """Per call of the case: its problems (m, n, k, alpha, beta); the layer of an moe case takes two calls."""
    kind = c["kind"]
    if kind in ("group", "shared"):
        one = (c["m"], c["n"], c["k"], c["alpha"], c["beta"])
        return [[one] * c["g"] + [one[:2] + (c["long_k"],) + one[3:]] * c.get("long_g", 0)] if c.get("long_k") else [[one] * c["g"]]
    if kind == "ragged":
        r = random.Random(c["shape_seed"])
        zero = set(r.sample(range(c["g"]), c["g"] // 16))
        return [[(_lu(r, c["mn_lo"], c["mn_hi"]), _lu(r, c["mn_lo"], c["mn_hi"]), _lu(r, c["k_lo"], c["k_hi"]),
                  0.0 if i in zero else r.uniform(-2.0, 2.0), r.uniform(-1.0, 1.0)) for i in range(c["g"])]]
    if kind == "moe":
        ex, _ = moe_ffn.route(c["tokens"], c["experts"], c["topk"], 1.0, np.random.default_rng(c["shape_seed"]))
        rows = np.bincount(ex.reshape(-1), minlength=c["experts"])
        return [[(int(r), c["f"], c["d"], 1.0, 0.0) for r in rows], [(int(r), c["d"], c["f"], 1.0, 0.0) for r in rows]]
    size, cols, _ = block_sparse.structure(c["atoms"], 0.1, c["cutoff"], c["basis"], np.random.default_rng(c["shape_seed"]))
    return [[(int(size[i]), c["nrhs"], int(size[j].sum()), 1.0, 0.0) for i, j in enumerate(cols)]]


def _offsets(counts):
    """256-byte aligned starts of consecutive blocks of doubles, and the total."""
    at = np.concatenate([[0], np.cumsum([(x + 31) // 32 * 32 for x in counts])]).astype(np.int64)
    return at[:-1].tolist(), max(32, int(at[-1]))


def _values(gen, count, phi, bad=0.0):
    """(U - 1/2) exp(phi Z), or U(-1, 1) for phi = 0; a share `bad` of NaN / +Inf / -Inf."""
    v = torch.rand(count, dtype=torch.float64, device="cuda", generator=gen)
    if phi == 0.0:
        v.mul_(2.0).sub_(1.0)
    else:
        v.sub_(0.5)
        for s in v.split(1 << 27):
            s.mul_(torch.randn(s.numel(), dtype=torch.float64, device="cuda", generator=gen).mul_(phi).exp_())
    if bad:
        vals = torch.tensor([float("nan"), float("inf"), float("-inf")], dtype=torch.float64, device="cuda")
        for s in v.split(1 << 27):
            at = torch.rand(s.numel(), device="cuda", generator=gen) < bad
            kind = torch.randint(0, 3, (int(at.sum()),), device="cuda", generator=gen)
            s[at] = vals[kind]
    return v


class _Call:
    """One grouped call: flat operands and the problem array."""

    def __init__(self, c, shapes, gen):
        self.shapes = shapes
        one_a = c["kind"] == "shared"
        self.oa, na = _offsets([m * k for m, n, k, *_ in (shapes[:1] if one_a else shapes)])
        if one_a:
            self.oa = self.oa * len(shapes)
        self.ob, nb = _offsets([k * n for m, n, k, *_ in shapes])
        self.oc, nc = _offsets([m * n for m, n, *_ in shapes])
        self.A = _values(gen, na, c["phi"], c["bad"])
        self.B = _values(gen, nb, c["phi"], c["bad"])
        self.C = [_values(gen, nc, 0.0) for _ in range(2 if c["api"] == "plan" else 1)]
        self.num = len(shapes)
        self.arr = self.problems(self.C[0])

    def problems(self, out):
        a, b, o = self.A.data_ptr(), self.B.data_ptr(), out.data_ptr()
        return G.problems_array([G.Problem(m, n, k, a + 8 * self.oa[i], max(1, m), b + 8 * self.ob[i], max(1, k),
                                           o + 8 * self.oc[i], max(1, m), al, be)
                                 for i, (m, n, k, al, be) in enumerate(self.shapes)])

    def pointers(self, out):
        p = lambda t, off: (C.c_void_p * self.num)(*[t.data_ptr() + 8 * x for x in off])  # noqa: E731
        return p(self.A, self.oa), p(self.B, self.ob), p(out, self.oc)


class _State:
    def __init__(self, c, seed):
        gen = torch.Generator(device="cuda")
        gen.manual_seed(int(seed))
        self.calls = [_Call(c, s, gen) for s in _shapes(c)]
        self.path = PATHS[c["path"]]
        self.cfg = G.Config(c["moduli"], 1e-15, 1, REPAIR[c["repair"]])
        self.api, self.handle, self.plan, self.step = c["api"], None, None, 0
        if self.api != "noalloc":
            cap = [max(sum(f(s) for s in call.shapes) for call in self.calls) + 1
                   for f in (lambda s: s[0] * s[2], lambda s: s[2] * s[1], lambda s: s[0] * s[1])]
            ks = [s[2] for call in self.calls for s in call.shapes if s[2] > 0]
            self.handle = G.Handle(max(call.num for call in self.calls), *cap, min_k=min(ks + [32]))
        if self.api == "plan":
            call, err = self.calls[0], C.c_int(0)
            self.plan = G.lib().ggemm_make_plan_ex(self.handle.h, self.path, C.byref(self.cfg), call.arr, call.num, C.byref(err))
            if not self.plan:
                raise RuntimeError(f"ggemm_make_plan_ex: {err.value}")
            self.ptrs = [call.pointers(o) for o in call.C]

    def __del__(self):
        if getattr(self, "plan", None):
            torch.cuda.synchronize()
            G.lib().ggemm_destroy_plan(self.plan)
        if getattr(self, "handle", None):
            self.handle.close()


def prepare(case, seed):
    return _State(case, seed)


def run(state):
    L = G.lib()
    if state.api == "plan":
        at = state.step & 1
        state.step += 1
        G.check(L.ggemm_plan_update_pointers(state.plan, *state.ptrs[at]), "ggemm_plan_update_pointers")
        G.check(L.ggemm_execute_plan(state.plan, None), "ggemm_execute_plan")
        return [state.calls[0].C[at]]
    for call in state.calls:
        if state.api == "noalloc":
            rc = L.ggemm_grouped_dgemm_noalloc(state.path, C.byref(state.cfg), call.arr, call.num, None, None)
        else:
            rc = L.ggemm_grouped_dgemm(state.handle.h, state.path, C.byref(state.cfg), call.arr, call.num, None)
        G.check(rc, "ggemm_grouped_dgemm")
    return [call.C[0] for call in state.calls]


def work(case):
    """Operands read once, C written once (and read when beta != 0); 2 m n k operations."""
    nbytes, flops = 0.0, 0.0
    for shapes in _shapes(case):
        for i, (m, n, k, alpha, beta) in enumerate(shapes):
            nbytes += 8.0 * m * n * (2 if beta != 0.0 else 1)
            if alpha != 0.0:
                nbytes += 8.0 * (k * n + (m * k if case["kind"] != "shared" or i == 0 else 0))
                flops += 2.0 * m * n * k
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # An emulated product is defined bit for bit (integer residue products, exact CRT, certificate
    # and repair in a fixed order), and the emulated paths take no other route for these cases.
    # Natively routed ones are FP64 sums in any order: against another library's order they measured
    # 1e-15 apart (2-norm) at k = 1024 and 2.8e-15 at k = 60000; four times the latter, with single
    # entries 40 times that over the root mean square.
    if case["path"] in ("emu", "reuse"):
        return "exact"
    return {"rel": 1.2e-14, "max": 4.8e-13}


def exact(case, seed):
    st = _State(dict(case, api="call"), seed)
    out = []
    for call in st.calls:
        o = call.C[0].clone()
        for i, (m, n, k, alpha, beta) in enumerate(call.shapes):
            if m == 0 or n == 0:
                continue
            at = call.oc[i]
            c0 = o[at:at + m * n].view(n, m)
            r = c0 * beta if beta != 0.0 else torch.zeros_like(c0)
            if alpha != 0.0 and k > 0:
                a = call.A[call.oa[i]:call.oa[i] + m * k].view(k, m)
                b = call.B[call.ob[i]:call.ob[i] + k * n].view(n, k)
                r = r + alpha * torch.matmul(b, a)
            o[at:at + m * n] = r.reshape(-1)
        out.append(o)
    return out
