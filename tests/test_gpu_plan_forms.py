"""GPU tests of the forms that a plan's stages take by launch size, knob and
register radix: every form's residues are the oracle's."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpu-resident-library_amd"))

from common import make_params  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import gpufhe
    return gpufhe


def rand_rows(mods, n, rng):
    return np.concatenate([rng.integers(0, int(m), n, dtype=np.uint64) for m in mods])


class Setup:
    def __init__(self, G, n, L, dnum, nkeys=1, knobs=(), **params):
        self.G, self.n, self.L = G, n, L
        self.P = make_params(n, L, dnum, **params)
        self.rng = np.random.default_rng(7 * n + 100 * L + dnum)
        self.ctx = G.Context(n, self.P.q, self.P.p, self.P.roots, dnum)
        for k, v in dict(knobs).items():
            self.ctx.set_knob(k, v)
        self.hk = [tuple(np.concatenate([rand_rows(self.P.mods, n, self.rng) for _ in range(self.P.dnum)])
                         for _ in range(2)) for _ in range(nkeys)]
        self.keys = [G.Key(self.ctx, av, bv, self.P.dnum) for av, bv in self.hk]
        self.s = G.Stream()

    def ct(self, level):
        return rand_rows(self.P.q[:level], self.n, self.rng)


def test_tuner_times_every_radix(G):
    """Radix 2^4, the fastest for large launches of whole transforms, is among
    the radices that the tuner times, and plans run at the one it chose."""
    P = make_params(1 << 14, 4, 2)
    ctx = G.Context(1 << 14, P.q, P.p, P.roots, 2)
    s = G.Stream()
    ctx.autotune(s, 2)
    rep = ctx.tuning_report()["ntt_radix"]
    assert set(rep["ms_per_fwd_inv_pass"]) == {"2", "3", "4"}, rep
    assert rep["chosen"] == ctx.ntt_radix()


# a ring of two 4096-element tiles per tower and the largest one; counts on
# both sides of the column and row passes' tile lines
@pytest.mark.parametrize("n,L,counts", [(1 << 13, 6, (1, 20, 130)), (1 << 17, 2, (1, 18))])
def test_whole_transforms_at_every_radix(G, n, L, counts):
    """The unfused schedule (whole transforms) at every register radix, in
    launches on small and on large tiles, over moduli of 50 and 60 bits."""
    t = Setup(G, n, L, 1)
    t.ctx.set_fusion(False)
    c = [[t.ct(L) for _ in range(4)] for _ in range(3)]
    d = [[G.Dev.of(x) for x in v] for v in c]
    w = [t.P.evalmult_rescale(L, *v, *t.hk[0]) for v in c]
    big = max(counts)
    o = [[G.Dev((L - 1) * n) for _ in range(2)] for _ in range(big)]
    ws = [t.ctx.workspace() for _ in range(big)]
    for radix in (2, 3, 4):
        t.ctx.set_ntt_radix(radix)
        for count in counts:
            plan = G.plan_evalmult_rescale(t.ctx, t.keys[0], [L] * count,
                                           *[[d[i % 3][j].ptr for i in range(count)] for j in range(4)],
                                           [x[0].ptr for x in o[:count]], [x[1].ptr for x in o[:count]], [x.ptr for x in ws[:count]])
            assert {"ntt_fwd", "ntt_inv"} <= {k for k, _ in plan.steps()}, plan.steps()
            plan.run(t.s)
            t.s.sync()
            for i in range(count):
                for k in range(2):
                    assert np.array_equal(o[i][k].download(), w[i % 3][k]), (radix, count, i, k)


@pytest.mark.parametrize("f64", [0, 1])
@pytest.mark.parametrize("dnum,down", [(1, "both"), (1, "modup"), (3, "both"), (3, "moddown")])
def test_stages_below_modup_min_wgs_run_apart(G, dnum, down, f64):
    """Fused ModUp and ModDown stages of fewer workgroups than modup_min_wgs run
    as transforms and conversions of their own: both stages, or only the one
    with fewer jobs (one part per operation against two components, or three
    parts against two).  Products, rotations (apart and over their inputs),
    hoisted rotations, keyswitches and linear transforms."""
    n, L, count = 1 << 14, 6, 8
    t = Setup(G, n, L, dnum, nkeys=2, knobs=dict(modup_f64=f64))
    P, ctx, s = t.P, t.ctx, t.s
    ks = [pow(5, 9, 2 * n), 2 * n - 1]
    c = [[t.ct(L) for _ in range(4)] for _ in range(count)]
    ws = [ctx.workspace() for _ in range(3 * count)]
    wp = [w.ptr for w in ws]
    some = (0, 1, count - 1)

    def fresh():
        return [[G.Dev.of(x) for x in v] for v in c]

    def col(d, j):
        return [x[j].ptr for x in d]

    def line(ups, downs):
        """the knob between the two stages' workgroups (ups parts, downs components)"""
        if down == "both":
            ctx.set_knob("modup_min_wgs", 1 << 30)
        else:
            lo, hi = (ups, downs) if down == "modup" else (downs, ups)
            if lo >= hi:
                return False
            ctx.set_knob("modup_min_wgs", lo * n // 1024 + 1)
        return True

    def run(plan, fused_down):
        kinds = [k for k, _ in plan.steps()]
        assert ("modup" in kinds) == (down == "moddown"), kinds
        assert (fused_down in kinds) == (down == "modup"), kinds
        plan.run(s)
        s.sync()

    def check(dev, want, what):
        assert np.array_equal(dev[0].download(want[0].size), want[0]), what
        assert np.array_equal(dev[1].download(want[1].size), want[1]), what

    assert line(count * dnum, 2 * count)
    for over in (False, True):
        d = fresh()
        o = [x[:2] for x in d] if over else [[G.Dev((L - 1) * n) for _ in range(2)] for _ in range(count)]
        run(G.plan_evalmult_rescale(ctx, t.keys[0], [L] * count, *[col(d, j) for j in range(4)], col(o, 0), col(o, 1), wp[:count]),
            "moddown")
        for i in some:
            check(o[i], P.evalmult_rescale(L, *c[i], *t.hk[0]), ("mult", over, i))
        d = fresh()
        o = [x[:2] for x in d] if over else [[G.Dev(L * n) for _ in range(2)] for _ in range(count)]
        kk, kh = [ks[i % 2] for i in range(count)], [t.keys[i % 2] for i in range(count)]
        run(G.plan_rotate(ctx, kh, [L] * count, kk, col(d, 0), col(d, 1), col(o, 0), col(o, 1), wp[:count]), "ksdown")
        for i in some:
            check(o[i], P.rotate(L, c[i][0], c[i][1], kk[i], *t.hk[i % 2]), ("rot", over, i))
        if line(count * dnum, 4 * count):
            d = fresh()
            h = [[G.Dev(L * n) for _ in range(2)] for _ in range(2 * count)]
            if over:   # the first rotation of each over its input
                for i in range(count):
                    h[2 * i] = d[i][:2]
            run(G.plan_rotate_hoisted(ctx, [L] * count, col(d, 0), col(d, 1), t.keys, ks, col(h, 0), col(h, 1), wp[:count], wp[count:]),
                "ksdown")
            for i in some:
                for j, w in enumerate(P.rotate_hoisted(L, c[i][0], c[i][1], ks, t.hk)):
                    check(h[2 * i + j], w, ("hoist", over, i, j))
        line(count * dnum, 2 * count)
    assert line(dnum, 2)
    d = fresh()
    o = [G.Dev(L * n) for _ in range(2)]
    G.check(G.lib.gf_keyswitch(ctx.h, t.keys[0].h, L, d[0][0].ptr, o[0].ptr, o[1].ptr, wp[0], s.s))
    s.sync()
    check(o, P.keyswitch(L, c[0][0], *t.hk[0]), "ks")
    G.check(G.lib.gf_evalmult(ctx.h, t.keys[0].h, L, *[x.ptr for x in d[0]], o[0].ptr, o[1].ptr, wp[0], s.s))
    s.sync()
    check(o, P.evalmult(L, *c[0], *t.hk[0]), "evalmult")
    pts = [t.ct(L) for _ in range(3)]
    dp = [G.Dev.of(x) for x in pts]
    G.linear_transform(ctx, L, d[0][0].ptr, d[0][1].ptr, [None] + t.keys, [1] + ks, [x.ptr for x in dp], o[0].ptr, o[1].ptr,
                       wp[0], wp[1:4], s)
    s.sync()
    check(o, P.linear_transform(L, c[0][0], c[0][1], [1] + ks, [None] + t.hk, pts), "linear")


@pytest.mark.parametrize("n,L,dnum,count", [(1 << 15, 6, 3, 17), (1 << 15, 7, 7, 14), (1 << 16, 5, 5, 11)])
def test_inner_products_on_large_tiles(G, n, L, dnum, count):
    """With a 61-bit modulus (inner products stored, integer rows) at radix 2^4,
    launches on both sides of the inner product's tile line: products and
    rotations of 3, 5 and 7 parts."""
    t = Setup(G, n, L, dnum, nkeys=1, q0bits=61)
    t.ctx.set_ntt_radix(4)
    c = [[t.ct(L) for _ in range(4)] for _ in range(2)]
    d = [[G.Dev.of(x) for x in v] for v in c]
    wm = [t.P.evalmult_rescale(L, *v, *t.hk[0]) for v in c]
    k = pow(5, 17, 2 * n)
    wr = [t.P.rotate(L, v[0], v[1], k, *t.hk[0]) for v in c]
    o = [[G.Dev(L * n) for _ in range(2)] for _ in range(count)]
    keep = [t.ctx.workspace() for _ in range(count)]
    ws = [w.ptr for w in keep]
    for cnt in (1, count):
        assert (cnt * L * n // 1024 >= 3072) == (cnt > 1)   # the Q rows' workgroups
        col = [[d[i % 2][j].ptr for i in range(cnt)] for j in range(4)]
        out = [[x[j].ptr for x in o[:cnt]] for j in range(2)]
        for plan, want in ((G.plan_evalmult_rescale(t.ctx, t.keys[0], [L] * cnt, *col, *out, ws[:cnt]), wm),
                           (G.plan_rotate(t.ctx, [t.keys[0]] * cnt, [L] * cnt, [k] * cnt, col[0], col[1], *out, ws[:cnt]), wr)):
            assert "ksi" in {x for x, _ in plan.steps()}, plan.steps()
            plan.run(t.s)
            t.s.sync()
            for i in range(cnt):
                for j in range(2):
                    assert np.array_equal(o[i][j].download(want[i % 2][j].size), want[i % 2][j]), (cnt, i, j)


# knobs that differ from the defaults
LAST_STEP = [dict(), dict(ntt_radix=2), dict(ntt_radix=4), dict(ksi_fin=0), dict(ksi_tensor=0), dict(ksi_tensor=0, ntt_radix=2),
             dict(modup_f64=0), dict(modup_f64=0, ntt_radix=2), dict(ksi_f64=0, ksi_extra=1), dict(ksi_rowpass=0),
             dict(ksi_rowpass=0, ntt_radix=2, ksi_f64=0), dict(tensor_ib=0), dict(ksi_extra=1, ntt_radix=2), dict(ksi_fin=0, ksi_extra=1),
             dict(moddown_fused=0), dict(modup_fused=0, ntt_radix=2)]
DEFAULTS = dict(ntt_radix=3, ksi_fin=1, ksi_tensor=1, modup_f64=1, ksi_f64=1, ksi_extra=0, ksi_rowpass=1, tensor_ib=1,
                moddown_fused=1, modup_fused=1)


@pytest.mark.parametrize("n,L,dnum,count", [(1 << 13, 6, 3, 24), (1 << 13, 8, 4, 16), (1 << 14, 6, 6, 8), (1 << 15, 5, 5, 5)])
def test_last_step_at_every_knob(G, n, L, dnum, count):
    """Batches above the line from which the Q rows' inner products take the
    outputs' row passes with them (and form the tensor products there): every
    knob and radix that changes those launches, levels mixed, products,
    rotations and hoisted rotations, buffers at 16-byte and at 8-byte addresses."""
    t = Setup(G, n, L, dnum, nkeys=2)
    P, ctx, s = t.P, t.ctx, t.s
    lv = [L - i % 2 for i in range(max(count, 6))]
    c = [[t.ct(lv[i]) for _ in range(4)] for i in range(6)]   # taken in turn
    ks = [pow(5, 13, 2 * n), 2 * n - 1]
    wm = [P.evalmult_rescale(lv[i], *c[i], *t.hk[0]) for i in range(6)]
    wr = [P.rotate(lv[i], c[i][0], c[i][1], ks[i % 2], *t.hk[i % 2]) for i in range(6)]
    wh = P.rotate_hoisted(lv[0], c[0][0], c[0][1], ks, t.hk)
    lv = lv[:count]
    ws = [ctx.workspace() for _ in range(count)]
    wp = [w.ptr for w in ws]
    hc = count // 4   # ciphertexts of the hoisted rotations, two rotations each

    def place(x, odd):
        d = G.Dev(x.size + 2)
        d.upload(x, odd)
        return d

    for odd in (0, 1):
        d = [[place(x, odd) for x in v] for v in c]
        at = [[x.at(odd) for x in d[i % 6]] for i in range(count)]
        o = [[G.Dev(L * n + 2) for _ in range(2)] for _ in range(count)]
        oat = [[x.at(odd) for x in v] for v in o]
        for knobs in LAST_STEP if not odd else LAST_STEP[:2] + [dict(modup_f64=0)]:
            for k, v in {**DEFAULTS, **knobs}.items():
                ctx.set_knob(k, v)
            fused = knobs.get("moddown_fused", 1)

            def run(plan, last, want, what):
                kinds = [k for k, _ in plan.steps()]
                assert not fused or kinds[-1] == ("ksi" if last else "ntt_fwd_b"), (knobs, odd, kinds)
                plan.run(s)
                s.sync()
                for i, w in enumerate(want):
                    for j in range(2):
                        assert np.array_equal(o[i][j].download(w[j].size, odd), w[j]), (what, knobs, odd, i, j)

            fin = knobs.get("ksi_fin", 1)
            run(G.plan_evalmult_rescale(ctx, t.keys[0], lv, *[[x[j] for x in at] for j in range(4)],
                                        [x[0] for x in oat], [x[1] for x in oat], wp),
                fin and knobs.get("ksi_rowpass", 1), [wm[i % 6] for i in range(count)], "mult")
            run(G.plan_rotate(ctx, [t.keys[i % 2] for i in range(count)], lv, [ks[i % 2] for i in range(count)],
                              [x[0] for x in at], [x[1] for x in at], [x[0] for x in oat], [x[1] for x in oat], wp),
                fin, [wr[i % 6] for i in range(count)], "rot")
            run(G.plan_rotate_hoisted(ctx, [L] * hc, [at[0][0]] * hc, [at[0][1]] * hc, t.keys, ks,
                                      [x[0] for x in oat[:2 * hc]], [x[1] for x in oat[:2 * hc]], wp[:hc], wp[hc:3 * hc]),
                fin and 2 * hc * L * (n // 512) >= 1024, [wh[i % 2] for i in range(2 * hc)], "hoist")


def test_largest_plan_in_the_static_job_area(G):
    """The allocation-free EvalMult+Rescale at the most towers and digits that a
    context takes (256 towers, 16 digits of 16, 14 special primes): its plan of
    nearly 5000 transforms still fits the static job area."""
    n, L, dnum = 1 << 10, 256, 16
    t = Setup(G, n, L, dnum)
    assert t.P.K == 14
    c = [t.ct(L) for _ in range(4)]
    d = [G.Dev.of(x) for x in c]
    o = [G.Dev((L - 1) * n) for _ in range(2)]
    G.check(G.lib.gf_evalmult_rescale_noalloc(t.ctx.h, t.keys[0].h, L, *[x.ptr for x in d], o[0].ptr, o[1].ptr, t.s.s))
    t.s.sync()
    for x, w in zip(o, t.P.evalmult_rescale(L, *c, *t.hk[0])):
        assert np.array_equal(x.download(), w)
