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
