"""GPU tests of the fused forms of the keyswitch path (fused ModUp, fused
ModDown with its row-pass epilogue) at the sizes where they can go wrong:
smallest and largest two-phase rings, one-tower levels, partial digits,
in-place outputs.  Every result is a residue, compared with the oracle's."""
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
    def __init__(self, G, n, L, dnum, nkeys=1, **knobs):
        self.G, self.n, self.L = G, n, L
        self.P = make_params(n, L, dnum)
        self.rng = np.random.default_rng(n + 100 * L + dnum)
        self.ctx = G.Context(n, self.P.q, self.P.p, self.P.roots, dnum)
        for k, v in knobs.items():
            self.ctx.set_knob(k, v)
        self.hk = [tuple(np.concatenate([rand_rows(self.P.mods, n, self.rng) for _ in range(self.P.dnum)])
                         for _ in range(2)) for _ in range(nkeys)]
        self.keys = [G.Key(self.ctx, av, bv, self.P.dnum) for av, bv in self.hk]
        self.s = G.Stream()

    def ct(self, level):
        return rand_rows(self.P.q[:level], self.n, self.rng)


# n, L, dnum: every two-phase split, a digit of one tower, six towers per digit
FUSED = [(1 << 13, 3, 3), (1 << 13, 6, 1), (1 << 14, 7, 3), (1 << 15, 5, 2), (1 << 16, 4, 2)]


@pytest.mark.parametrize("f64", [0, 1])
@pytest.mark.parametrize("n,L,dnum", FUSED)
def test_fused_moddown_of_keyswitches(G, n, L, dnum, f64):
    """Keyswitch, EvalMult, rotation, hoisted rotations and the linear
    transform with the fused ModDown forced on for single operations, also
    with outputs over the inputs."""
    t = Setup(G, n, L, dnum, nkeys=2, modup_min_wgs=0, modup_f64=f64)
    P, ctx, s = t.P, t.ctx, t.s
    key, (av, bv) = t.keys[0], t.hk[0]
    ws = ctx.workspace()
    ks = [pow(5, 3, 2 * n), 2 * n - 1]
    for level in sorted({1, 2, L - 1, L}):
        c = [t.ct(level) for _ in range(4)]
        w = P.keyswitch(level, c[0], av, bv)
        for inplace in (False, True):
            d, b0, b1 = G.Dev.of(c[0]), G.Dev(level * n), G.Dev(level * n)
            if inplace:
                b0 = d
            G.check(G.lib.gf_keyswitch(ctx.h, key.h, level, d.ptr, b0.ptr, b1.ptr, ws.ptr, s.s))
            s.sync()
            assert np.array_equal(b0.download(), w[0]) and np.array_equal(b1.download(), w[1]), ("ks", level, inplace)
        w = P.evalmult(level, *c, av, bv)
        d = [G.Dev.of(x) for x in c]
        o = [G.Dev(level * n) for _ in range(2)]
        G.check(G.lib.gf_evalmult(ctx.h, key.h, level, *[x.ptr for x in d], o[0].ptr, o[1].ptr, ws.ptr, s.s))
        s.sync()
        assert np.array_equal(o[0].download(), w[0]) and np.array_equal(o[1].download(), w[1]), ("mult", level)
        w = P.rotate(level, c[0], c[1], ks[0], av, bv)
        for inplace in (False, True):
            d = [G.Dev.of(x) for x in c[:2]]
            o = d if inplace else [G.Dev(level * n) for _ in range(2)]
            G.check(G.lib.gf_rotate(ctx.h, key.h, level, ks[0], d[0].ptr, d[1].ptr, o[0].ptr, o[1].ptr, ws.ptr, s.s))
            s.sync()
            assert np.array_equal(o[0].download(), w[0]) and np.array_equal(o[1].download(), w[1]), ("rot", level, inplace)
    level = L
    wr = [ctx.workspace() for _ in range(3)]
    c = [t.ct(level) for _ in range(2)]
    d = [G.Dev.of(x) for x in c]
    o = [[G.Dev(level * n) for _ in range(2)] for _ in range(2)]
    G.rotate_hoisted(ctx, level, d[0].ptr, d[1].ptr, t.keys, ks, [x[0].ptr for x in o], [x[1].ptr for x in o], ws.ptr,
                     [x.ptr for x in wr[:2]], s)
    s.sync()
    for (w0, w1), x in zip(P.rotate_hoisted(level, c[0], c[1], ks, t.hk), o):
        assert np.array_equal(x[0].download(), w0) and np.array_equal(x[1].download(), w1), "hoisted"
    pts = [t.ct(level) for _ in range(3)]
    dp = [G.Dev.of(x) for x in pts]
    a = [G.Dev(level * n) for _ in range(2)]
    G.linear_transform(ctx, level, d[0].ptr, d[1].ptr, [None] + t.keys, [1] + ks, [x.ptr for x in dp], a[0].ptr, a[1].ptr,
                       ws.ptr, [x.ptr for x in wr], s)
    s.sync()
    w0, w1 = P.linear_transform(level, c[0], c[1], [1] + ks, [None] + t.hk, pts)
    assert np.array_equal(a[0].download(), w0) and np.array_equal(a[1].download(), w1), "linear"


@pytest.mark.parametrize("split", [1, 1 << 20])
@pytest.mark.parametrize("n,L,dnum", [(1 << 13, 7, 2), (1 << 14, 5, 5), (1 << 15, 8, 2)])
def test_uneven_batch_in_one_launch(G, n, L, dnum, split):
    """EvalMult+Rescale, rotations and hoisted rotations of every level in one
    plan: parts of every source count share a launch, with each job's targets
    in one workgroup (split 1) and one workgroup per target (2^20)."""
    t = Setup(G, n, L, dnum, nkeys=2, modup_min_wgs=0, modup_split_wgs=split)
    P, ctx, s = t.P, t.ctx, t.s
    ks = [pow(5, 7, 2 * n), 3]
    levels = list(range(2, L + 1))
    c = [[t.ct(lv) for _ in range(4)] for lv in levels]
    d = [[G.Dev.of(x) for x in v] for v in c]
    ws = [ctx.workspace() for _ in range(3 * len(levels))]
    o = [[G.Dev((lv - 1) * n) for _ in range(2)] for lv in levels]
    plan = G.plan_evalmult_rescale(ctx, t.keys[0], levels, *[[x[j].ptr for x in d] for j in range(4)],
                                   [x[0].ptr for x in o], [x[1].ptr for x in o], [w.ptr for w in ws[:len(levels)]])
    r = [[G.Dev(lv * n) for _ in range(2)] for lv in levels]
    rplan = G.plan_rotate(ctx, [t.keys[i % 2] for i in range(len(levels))], levels, [ks[i % 2] for i in range(len(levels))],
                          [x[0].ptr for x in d], [x[1].ptr for x in d], [x[0].ptr for x in r], [x[1].ptr for x in r],
                          [w.ptr for w in ws[:len(levels)]])
    h = [[G.Dev(lv * n) for _ in range(2)] for lv in levels for _ in ks]
    hplan = G.plan_rotate_hoisted(ctx, levels, [x[0].ptr for x in d], [x[1].ptr for x in d], t.keys, ks,
                                  [x[0].ptr for x in h], [x[1].ptr for x in h], [w.ptr for w in ws[:len(levels)]],
                                  [w.ptr for w in ws[len(levels):]])
    for p in (plan, rplan, hplan):
        p.run(s)
    s.sync()
    for i, lv in enumerate(levels):
        w = P.evalmult_rescale(lv, *c[i], *t.hk[0])
        assert np.array_equal(o[i][0].download(), w[0]) and np.array_equal(o[i][1].download(), w[1]), ("mult", lv)
        w = P.rotate(lv, c[i][0], c[i][1], ks[i % 2], *t.hk[i % 2])
        assert np.array_equal(r[i][0].download(), w[0]) and np.array_equal(r[i][1].download(), w[1]), ("rot", lv)
        for j, w in enumerate(P.rotate_hoisted(lv, c[i][0], c[i][1], ks, t.hk)):
            x = h[2 * i + j]
            assert np.array_equal(x[0].download(), w[0]) and np.array_equal(x[1].download(), w[1]), ("hoist", lv, j)


@pytest.mark.parametrize("n,L,dnum", [(1 << 13, 6, 2), (1 << 14, 5, 1), (1 << 16, 9, 1), (1 << 17, 4, 1)])
def test_column_pass_tiles(G, n, L, dnum):
    """Whole transforms (fused ModUp and ModDown off) in launches on both sides
    of the column tile's line: a few towers, and enough to fill the chip."""
    t = Setup(G, n, L, dnum, modup_fused=0, moddown_fused=0)
    ws = t.ctx.workspace()
    for level in (1, L):
        d = t.ct(level)
        w = t.P.keyswitch(level, d, *t.hk[0])
        x, b0, b1 = G.Dev.of(d), G.Dev(level * n), G.Dev(level * n)
        G.check(G.lib.gf_keyswitch(t.ctx.h, t.keys[0].h, level, x.ptr, b0.ptr, b1.ptr, ws.ptr, t.s.s))
        t.s.sync()
        assert np.array_equal(b0.download(), w[0]) and np.array_equal(b1.download(), w[1]), level


@pytest.mark.parametrize("f64", [0, 1])
@pytest.mark.parametrize("n,L,dnum,count", [(1 << 13, 6, 2, 16), (1 << 13, 7, 7, 12), (1 << 14, 6, 6, 8), (1 << 16, 5, 1, 3)])
def test_last_step_in_the_inner_product(G, n, L, dnum, count, f64):
    """Batches large enough that the Q rows' inner products take the outputs'
    row passes with them, 1 to 7 parts (7 transform more rows than fit), and
    rotations read their inputs through the automorphism; rotations whose
    outputs are their own or another's inputs take permuted copies instead."""
    t = Setup(G, n, L, dnum, nkeys=2, modup_f64=f64)
    P, ctx, s = t.P, t.ctx, t.s
    ks = [pow(5, 11, 2 * n), 2 * n - 1]
    c = [[t.ct(L) for _ in range(4)] for _ in range(count)]
    ws = [ctx.workspace() for _ in range(3 * count)]
    wp = [w.ptr for w in ws]

    def fresh():
        return [[G.Dev.of(x) for x in v] for v in c]

    def col(d, j):
        return [x[j].ptr for x in d]

    def check(dev, want, what):
        assert np.array_equal(dev[0].download(want[0].size), want[0]), what
        assert np.array_equal(dev[1].download(want[1].size), want[1]), what

    last = "ksi" if dnum < 7 else "ntt_fwd_b"
    some = sorted({0, 1, count - 1})
    d = fresh()
    o = [[G.Dev((L - 1) * n) for _ in range(2)] for _ in range(count)]
    plan = G.plan_evalmult_rescale(ctx, t.keys[0], [L] * count, *[col(d, j) for j in range(4)], col(o, 0), col(o, 1), wp[:count])
    assert plan.steps()[-1][0] == last, plan.steps()
    plan.run_graph(s)
    s.sync()
    for i in some:
        check(o[i], P.evalmult_rescale(L, *c[i], *t.hk[0]), ("mult", i))
    # a product over its own first factor, then over the next one's
    for shift in (0, 1):
        d = fresh()
        o = [d[(i + shift) % count][:2] for i in range(count)]
        plan = G.plan_evalmult_rescale(ctx, t.keys[0], [L] * count, *[col(d, j) for j in range(4)], col(o, 0), col(o, 1), wp[:count])
        plan.run(s)
        s.sync()
        for i in some:
            check(o[i], P.evalmult_rescale(L, *c[i], *t.hk[0]), ("mult over an input", shift, i))
    kk, kh = [ks[i % 2] for i in range(count)], [t.keys[i % 2] for i in range(count)]
    rot = {i: P.rotate(L, c[i][0], c[i][1], kk[i], *t.hk[i % 2]) for i in some}
    # apart; in place; every output over the next one's input
    for shift in (None, 0, 1):
        d = fresh()
        o = [[G.Dev(L * n) for _ in range(2)] for _ in range(count)]
        if shift is not None:
            o = [d[(i + shift) % count] for i in range(count)]
        plan = G.plan_rotate(ctx, kh, [L] * count, kk, col(d, 0), col(d, 1), col(o, 0), col(o, 1), wp[:count])
        kinds = [k for k, _ in plan.steps()]
        assert ("perm" in kinds) == (shift is not None) and kinds[-1] == (last if shift is None else "ntt_fwd_b"), kinds
        plan.run(s)
        s.sync()
        for i in some:
            check(o[i], rot[i], ("rot", shift, i))
    d = fresh()
    h = [[G.Dev(L * n) for _ in range(2)] for _ in range(2 * count)]
    plan = G.plan_rotate_hoisted(ctx, [L] * count, col(d, 0), col(d, 1), t.keys, ks, col(h, 0), col(h, 1), wp[:count], wp[count:])
    assert plan.steps()[-1][0] == "ksi", plan.steps()
    plan.run(s)
    s.sync()
    for i in some:
        for j, w in enumerate(P.rotate_hoisted(L, c[i][0], c[i][1], ks, t.hk)):
            check(h[2 * i + j], w, ("hoist", i, j))


@pytest.mark.parametrize("f64", [0, 1])
@pytest.mark.parametrize("n,L,ascending", [(1 << 13, 2, False), (1 << 14, 6, True), (1 << 15, 7, False), (1 << 16, 3, True),
                                           (1 << 17, 3, False)])
def test_fused_rescale(G, n, L, ascending, f64):
    """The rescale's fused form at every ring split, the dropped modulus below
    and above the others, two towers and more, one component in place."""
    import oracle as O
    P = make_params(n, L, 1)
    if ascending:
        q = sorted(int(m) for m in P.q)
        roots = [int(O.lib.or_native_root(n, m)) for m in q + [int(m) for m in P.p]]
        P = O.Params(n, q, P.p, roots, 1)
    ctx = G.Context(n, P.q, P.p, P.roots, 1)
    ctx.set_knob("modup_f64", f64)
    rng, s = np.random.default_rng(n + L), G.Stream()
    ws, rs = ctx.workspace(), G.Dev(G.lib.gf_rescale_ws_bytes(ctx.h) // 8)
    for level in sorted({2, L}):
        c = [rand_rows(P.q[:level], n, rng) for _ in range(2)]
        w = [P.rescale(x, level) for x in c]
        d = [G.Dev.of(x) for x in c]
        o = [G.Dev((level - 1) * n) for _ in range(2)]
        G.check(G.lib.gf_rescale(ctx.h, level, d[0].ptr, d[1].ptr, o[0].ptr, o[1].ptr, ws.ptr, s.s))
        G.check(G.lib.gf_rescale_comp(ctx.h, level, d[1].ptr, d[1].ptr, rs.ptr, s.s))
        s.sync()
        assert np.array_equal(o[0].download(), w[0]) and np.array_equal(o[1].download(), w[1]), level
        assert np.array_equal(d[1].download((level - 1) * n), w[1]), ("in place", level)


@pytest.mark.parametrize("f64", [0, 1])
@pytest.mark.parametrize("n,L,dnum", [(1 << 13, 24, 2), (1 << 14, 14, 2), (1 << 15, 10, 1), (1 << 16, 8, 1), (1 << 17, 9, 1)])
def test_wide_digits(G, n, L, dnum, f64):
    """Digits of 7 to 12 towers and 6 to 11 special primes: the fused forms'
    widest sums, with levels whose digits hold few, six, seven and all towers."""
    t = Setup(G, n, L, dnum, modup_f64=f64)
    P, ctx, s = t.P, t.ctx, t.s
    alpha = -(-L // dnum)
    av, bv = t.hk[0]
    ws = ctx.workspace()
    levels = sorted({2, 6, 7, alpha, L} if n < 1 << 16 else {7, L})
    for level in levels:
        c = [t.ct(level) for _ in range(4)]
        d = [G.Dev.of(x) for x in c]
        o = [G.Dev(level * n) for _ in range(2)]
        G.check(G.lib.gf_keyswitch(ctx.h, t.keys[0].h, level, d[0].ptr, o[0].ptr, o[1].ptr, ws.ptr, s.s))
        s.sync()
        w = P.keyswitch(level, c[0], av, bv)
        assert np.array_equal(o[0].download(), w[0]) and np.array_equal(o[1].download(), w[1]), ("ks", level)
        G.check(G.lib.gf_evalmult_rescale(ctx.h, t.keys[0].h, level, *[x.ptr for x in d], o[0].ptr, o[1].ptr, ws.ptr, s.s))
        s.sync()
        w = P.evalmult_rescale(level, *c, av, bv)
        m = (level - 1) * n
        assert np.array_equal(o[0].download(m), w[0]) and np.array_equal(o[1].download(m), w[1]), ("mult", level)
    if n < 1 << 16:   # every level in one plan: narrow and wide digits in one stage
        lv = list(range(2, L + 1))
        c = [[t.ct(x) for _ in range(4)] for x in lv]
        d = [[G.Dev.of(x) for x in v] for v in c]
        o = [[G.Dev((x - 1) * n) for _ in range(2)] for x in lv]
        wss = [ctx.workspace() for _ in lv]
        plan = G.plan_evalmult_rescale(ctx, t.keys[0], lv, *[[x[j].ptr for x in d] for j in range(4)], [x[0].ptr for x in o],
                                       [x[1].ptr for x in o], [w.ptr for w in wss])
        plan.run(s)
        s.sync()
        for i in (0, 4, 5, alpha - 2, len(lv) - 1):
            w = P.evalmult_rescale(lv[i], *c[i], av, bv)
            assert np.array_equal(o[i][0].download(), w[0]) and np.array_equal(o[i][1].download(), w[1]), ("batch", lv[i])


@pytest.mark.parametrize("f64", [0, 1])
@pytest.mark.parametrize("n,L,dnum,count", [(1 << 13, 8, 4, 24), (1 << 14, 5, 5, 12), (1 << 17, 4, 4, 4)])
def test_last_step_inputs_through_lds(G, n, L, dnum, count, f64):
    """Products of 4 and 5 parts, whose last step brings the input towers into
    LDS, beside products of fewer parts (levels below), which may share the
    launch: tiles at both ends of the ring, each output against the oracle's."""
    t = Setup(G, n, L, dnum, modup_f64=f64)
    lv = [L - 2 * (i % 2) for i in range(count)]
    c = [[t.ct(x) for _ in range(4)] for x in lv]
    d = [[G.Dev.of(x) for x in v] for v in c]
    o = [[G.Dev((x - 1) * n) for _ in range(2)] for x in lv]
    ws = [t.ctx.workspace() for _ in range(count)]
    plan = G.plan_evalmult_rescale(t.ctx, t.keys[0], lv, *[[x[j].ptr for x in d] for j in range(4)],
                                   [x[0].ptr for x in o], [x[1].ptr for x in o], [w.ptr for w in ws])
    assert plan.steps()[-1][0] == "ksi", plan.steps()
    plan.run(t.s)
    t.s.sync()
    for i in sorted({0, 1, count - 2, count - 1}):
        w = t.P.evalmult_rescale(lv[i], *c[i], *t.hk[0])
        assert np.array_equal(o[i][0].download(), w[0]) and np.array_equal(o[i][1].download(), w[1]), i
