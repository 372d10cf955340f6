"""CPU tests of the fused steps' further forms: tests/emu/emu_forms.cpp runs the
kernels' headers workgroup by workgroup, between guard words, and every result
is a residue compared with its definition over the oracle's transforms."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

import oracle as O

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
u64, u64p = C.c_uint64, C.POINTER(C.c_uint64)
KSI_PLAIN, KSI_FIN, KSI_FIN_TENSOR, KSI_FIN_TENSOR_IN = range(4)


class KsiArgs(C.Structure):
    _fields_ = [(k, u64) for k in ("n", "q", "rmax", "form", "np", "xf", "pairs", "f64", "gk")] + \
        [(k, u64p) for k in ("fw", "fwp", "iw", "iwp", "src", "kb", "ka", "o0", "o1", "v0", "v1", "e0", "e1")] + \
        [(k, u64) for k in ("ci", "ce", "e_plain")] + [("in_", u64p * 4)] + [(k, u64p) for k in ("d0", "d1")] + \
        [(k, u64) for k in ("dpinv", "post")]


pp = C.POINTER(u64p)


class ModupArgs(C.Structure):
    _fields_ = [(k, u64) for k in ("n", "sp", "sc", "rs", "f64", "c60", "len")] + \
        [("src", pp), ("sq", u64p), ("sw", pp), ("swp", pp), ("post", u64p), ("tq", u64p), ("tw", pp), ("twp", pp), ("tab", u64p),
         ("tabd", u64p), ("pinv", u64), ("s2", u64p), ("dst", u64p)]


@pytest.fixture(scope="module")
def emu(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ absent")
    so = str(tmp_path_factory.mktemp("emu") / "libemuforms.so")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-fPIC", "-shared",
                           "-I" + os.path.join(ROOT, "gpu-resident-library_amd", "csrc"),
                           "-o", so, os.path.join(HERE, "emu", "emu_forms.cpp")])
    lib = C.CDLL(so)
    lib.emu_ksi_form.argtypes = [C.POINTER(KsiArgs)]
    lib.emu_modup_form.argtypes = [C.POINTER(ModupArgs)]
    lib.emu_ntt_tiles.argtypes = [u64p, u64, u64, u64p, u64p, C.c_int, u64, C.c_int, u64]
    for f in (lib.emu_ksi_form, lib.emu_modup_form, lib.emu_ntt_tiles):
        f.restype = None
    return lib


def mulmod(a, b, q):
    return np.array(a.astype(object) * (b if isinstance(b, int) else b.astype(object)) % q, np.uint64)


def addmod(a, b, q):
    return np.array((a.astype(object) + b.astype(object)) % q, np.uint64)


def galois(x, k):
    """the evaluation-domain automorphism of index k (0: none), bit-reversed order"""
    if not k:
        return x
    n = x.size
    logn = n.bit_length() - 1
    brv = np.array([int(format(i, "0%db" % logn)[::-1], 2) for i in range(n)])
    e = (2 * brv + 1) * k % (2 * n)
    return x[brv[e >> 1]]


class Tables:
    def __init__(self, n, q, psi=None):
        self.q = q
        self.psi = int(O.lib.or_native_root(n, q)) if psi is None else psi
        self.fr, self.fp, self.ir, self.ip, self.ni, self.nip = O.root_tables(n, q, self.psi)

    def ntt(self, x):
        return O.ntt(x, self.q, self.fr, self.fp)

    def intt(self, x):
        return O.intt(x, self.q, self.ir, self.ip, self.ni, self.nip)


def uniform(rng, q, *shape):
    x = rng.integers(0, q, shape, dtype=np.uint64)
    x[..., :3] = q - 1
    return x


# transformed parts of 1 to 7 (the untransformed one, if any, at either end)
PARTS = [(1, 0b0), (1, 0b1), (2, 0b01), (3, 0b101), (4, 0b1110), (5, 0b11011), (6, 0b111101), (7, 0b1011111)]


@pytest.mark.parametrize("np_,xf", PARTS)
@pytest.mark.parametrize("logn", [13, 16])
def test_inner_product_forms(emu, logn, np_, xf):
    """sum_p digit_p key_p through every form of the fused step: stored; with the
    untransformed digits read through an automorphism; as the inverse transforms
    of the dropped tower t + sum P^-1; on tiles of 1024; with the last step's NTT(v) + sum ci + e
    (e times ce, as it is through the automorphism, or absent); and with e and
    the untransformed digit formed from two ciphertexts' rows, read or brought
    through LDS."""
    n = 1 << logn
    for bits in (50, 59, 61) if logn == 13 else (50,):
        q = int(O.native_primes(1, bits, n)[0])
        T = Tables(n, q)
        rng = np.random.default_rng(100 * logn + np_ + bits)
        src, kb, ka = (uniform(rng, q, np_, n) for _ in range(3))
        v, e, d = uniform(rng, q, 2, n), uniform(rng, q, 2, n), uniform(rng, q, 2, n)
        cts = uniform(rng, q, 4, n)
        ci, ce, dpinv = (int(rng.integers(1, q)) for _ in range(3))
        gk = pow(5, 21, 2 * n)
        Rinv = pow(1 << 64, -1, q)
        t0, t1 = mulmod(cts[0], cts[2], q), addmod(mulmod(cts[0], cts[3], q), mulmod(cts[1], cts[2], q), q)
        t2 = mulmod(cts[1], cts[3], q)
        dig = [T.ntt(src[p]) if (xf >> p) & 1 else None for p in range(np_)]

        def inner(plain):
            w = [np.zeros(n, object), np.zeros(n, object)]
            for p in range(np_):
                x = (plain(p) if dig[p] is None else dig[p]).astype(object)
                w[0] += x * kb[p].astype(object)
                w[1] += x * ka[p].astype(object)
            return [np.array(x * Rinv % q, np.uint64) for x in w]

        sums = {g: inner(lambda p: galois(src[p], g)) for g in (0, gk)}
        sums["tensor"] = inner(lambda p: t2)
        nv = [T.ntt(x) for x in v]
        post = int(T.ni)

        def run(form, rmax, pairs, f64, g=0, plain=0, es=(0, 1), drop=False):
            o = np.zeros((2, n), np.uint64)
            a = KsiArgs(n=n, q=q, rmax=rmax, form=form, np=np_, xf=xf, pairs=pairs, f64=f64, gk=g, ci=ci, ce=ce, e_plain=plain,
                        dpinv=dpinv, post=post)
            for k, x in dict(fw=T.fr, fwp=T.fp, iw=T.ir, iwp=T.ip, src=src, kb=kb, ka=ka, o0=o[0], o1=o[1], v0=v[0],
                             v1=v[1]).items():
                setattr(a, k, O.P(np.ascontiguousarray(x) if x.base is None else x))
            for k, j in (("e0", 0), ("e1", 1)):
                setattr(a, k, O.P(e[j]) if j in es else None)
            for j in range(4):
                a.in_[j] = O.P(cts[j])
            if drop:
                a.d0, a.d1 = O.P(d[0]), O.P(d[1])
            emu.emu_ksi_form(C.byref(a))
            return o

        for pairs in (0, 1):   # 1024-element tiles at radix 2^4
            o = run(KSI_PLAIN, 4, pairs, 0)
            assert np.array_equal(o[0], sums[0][0]) and np.array_equal(o[1], sums[0][1]), (bits, pairs)
        for rmax in (2, 3):
            for f64 in (0, 1) if bits == 50 else (0,):
                for pairs in (0, 1):
                    key = (bits, rmax, f64, pairs)
                    for g in (0, gk):
                        o = run(KSI_PLAIN, rmax, pairs, f64, g)
                        assert np.array_equal(o[0], sums[g][0]) and np.array_equal(o[1], sums[g][1]), key + (g,)
                    o = run(KSI_PLAIN, rmax, pairs, f64, drop=True)
                    for j in range(2):
                        w = T.intt(addmod(d[j], mulmod(sums[0][j], dpinv, q), q))
                        assert np.array_equal(o[j], w), key + ("drop", j)
                    if bin(xf).count("1") + 2 > 7:
                        continue
                    o = run(KSI_FIN, rmax, pairs, f64)
                    for j in range(2):
                        w = addmod(addmod(nv[j], mulmod(sums[0][j], ci, q), q), mulmod(e[j], ce, q), q)
                        assert np.array_equal(o[j], w), key + ("fin", j)
                    for es in ((0, 1), (0,), ()):
                        o = run(KSI_FIN, rmax, pairs, f64, gk, 1, es)
                        for j in range(2):
                            w = addmod(nv[j], mulmod(sums[gk][j], ci, q), q)
                            if j in es:
                                w = addmod(w, galois(e[j], gk), q)
                            assert np.array_equal(o[j], w), key + ("fin plain", es, j)
                    if not pairs or np_ > 6 or bits > 60 or bin(xf).count("1") != np_ - 1:
                        continue
                    for form in (KSI_FIN_TENSOR, KSI_FIN_TENSOR_IN):
                        o = run(form, rmax, pairs, f64)
                        for j, t in enumerate((t0, t1)):
                            w = addmod(addmod(nv[j], mulmod(sums["tensor"][j], ci, q), q), mulmod(t, ce, q), q)
                            assert np.array_equal(o[j], w), key + ("tensor", form, j)


def moduli(n, count60, count50):
    q = [int(x) for x in O.native_primes(count60, 60, n)]
    return q + [int(x) for x in O.native_primes(count50, 50, n, q)]


def ptrs(arrays):
    return (u64p * len(arrays))(*[O.P(a) for a in arrays])


@pytest.mark.parametrize("logn,sp,wide", [(13, 1, 1), (13, 6, 1), (13, 7, 1), (13, 7, 7), (13, 8, 2), (13, 9, 9), (13, 11, 3),
                                          (13, 12, 12), (13, 12, 1), (16, 7, 1), (16, 12, 12)])
def test_modup_of_many_sources(emu, logn, sp, wide):
    """The fused ModUp over 1, 6 and 7 to 12 sources, `wide` of them of 60 bits
    (the largest sums), to targets of 60 and 50 bits in ranges of one and of
    all: sum_i INTT(x_i) f_i tab_i R^-1 mod t, transformed, with integer and
    with fp64 passes and, where it applies, the R = 2^60 reduction."""
    n = 1 << logn
    mods = moduli(n, wide + 1, sp - wide + 2)
    sm, tm = mods[:wide] + mods[wide + 1:wide + 1 + sp - wide], [mods[wide]] + mods[-2:]
    rng = np.random.default_rng(logn * 100 + sp + wide)
    S, TT = [Tables(n, q) for q in sm], [Tables(n, q) for q in tm]
    x = [uniform(rng, q, n) for q in sm]
    f = [int(rng.integers(1, q)) for q in sm]
    tab = np.array([int(rng.integers(0, t)) for _ in range(sp) for t in tm], np.uint64)
    tab[:3] = [t - 1 for t in tm]
    co = [mulmod(s.intt(a), v, s.q).astype(object) for s, a, v in zip(S, x, f)]
    post = O.U([v * int(s.ni) % s.q for v, s in zip(f, S)])
    for f64 in (0, 1):
        for c60 in (0, 1):
            if c60 and (sp > 6 or 5 * sum(sm) > 6 << 60):
                continue
            Rinv = [pow(1 << (60 if c60 else 64), -1, t) for t in tm]
            want = [tt.ntt(np.array(sum(c * int(tab[i * 3 + j]) for i, c in enumerate(co)) % t * Rinv[j] % t, np.uint64))
                    for j, (t, tt) in enumerate(zip(tm, TT))]
            for ln in (1, 3):
                dst = np.zeros(3 * n, np.uint64)
                sqv, tqv = O.U(sm), O.U(tm)
                a = ModupArgs(n=n, sp=sp, sc=3, rs=0, f64=f64, c60=c60, len=ln, src=ptrs(x), sq=O.P(sqv),
                              sw=ptrs([s.ir for s in S]), swp=ptrs([s.ip for s in S]), post=O.P(post), tq=O.P(tqv),
                              tw=ptrs([s.fr for s in TT]), twp=ptrs([s.fp for s in TT]), tab=O.P(tab), dst=O.P(dst))
                emu.emu_modup_form(C.byref(a))
                for j in range(3):
                    assert np.array_equal(dst[j * n:(j + 1) * n], want[j]), (f64, c60, ln, j)


@pytest.mark.parametrize("logn,K", [(13, 0), (13, 1), (13, 6), (13, 7), (13, 8), (13, 11), (13, 12), (16, 0), (16, 12)])
def test_moddown_with_the_dropped_tower_as_a_source(emu, logn, K):
    """The fused ModDown's rescale mode over K special primes of 60 bits, the
    dropped tower one more source, larger and smaller than the targets (K = 0:
    a plain rescale): with dv = INTT(x_d) - pinv sum_k INTT(x_k) f_k tabd_k R^-1,
    centred, the targets' sum_k INTT(x_k) f_k tab_k R^-1 + s2 dv, transformed."""
    n = 1 << logn
    mods = moduli(n, K + 2, 4)
    pm, rest = mods[:K], mods[K:]
    for old in (rest[0], rest[2]):   # of 60 bits; of 50 bits, between the targets
        tm = [rest[1], rest[3], rest[4]] if old == rest[2] else [rest[1], rest[2], rest[5]]
        rng = np.random.default_rng(logn * 10 + K)
        sm = pm + [old]
        S, TT = [Tables(n, q) for q in sm], [Tables(n, q) for q in tm]
        x = [uniform(rng, q, n) for q in sm]
        f = [int(rng.integers(1, q)) for q in pm]
        tab = np.array([int(rng.integers(0, t)) for _ in range(K) for t in tm] + [0], np.uint64)
        tab[:3 if K else 0] = [t - 1 for t in tm][:3 if K else 0]
        tabd = np.array([int(rng.integers(0, old)) for _ in range(K)] + [0], np.uint64)
        s2 = O.U([int(rng.integers(1, t)) for t in tm])
        pinv = int(rng.integers(1, old))
        co = [mulmod(s.intt(a), v, s.q).astype(object) for s, a, v in zip(S, x, f)]
        dv = S[K].intt(x[K]).astype(object)
        if K:
            cd = sum(c * int(tabd[k]) for k, c in enumerate(co)) % old * pow(1 << 64, -1, old) % old
            dv = (dv - cd * pinv) % old
        dv = np.where(dv > old // 2, dv - old, dv)
        want = []
        for j, (t, tt) in enumerate(zip(tm, TT)):
            w = dv * int(s2[j])
            if K:
                w = w + sum(c * int(tab[k * 3 + j]) for k, c in enumerate(co)) % t * pow(1 << 64, -1, t)
            want.append(tt.ntt(np.array(w % t, np.uint64)))
        post = O.U([v * int(s.ni) % s.q for v, s in zip(f + [1], S)])
        for f64 in (0, 1):
            for ln in (1, 3):
                dst = np.zeros(3 * n, np.uint64)
                sqv, tqv = O.U(sm), O.U(tm)
                a = ModupArgs(n=n, sp=K, sc=3, rs=1, f64=f64, c60=0, len=ln, src=ptrs(x), sq=O.P(sqv),
                              sw=ptrs([s.ir for s in S]), swp=ptrs([s.ip for s in S]), post=O.P(post), tq=O.P(tqv),
                              tw=ptrs([s.fr for s in TT]), twp=ptrs([s.fp for s in TT]), tab=O.P(tab), tabd=O.P(tabd), pinv=pinv,
                              s2=O.P(s2), dst=O.P(dst))
                emu.emu_modup_form(C.byref(a))
                for j in range(3):
                    assert np.array_equal(dst[j * n:(j + 1) * n], want[j]), (old, f64, ln, j)


@pytest.mark.parametrize("logn", [13, 16])
@pytest.mark.parametrize("bits", [50, 58, 60])
def test_row_pass_on_large_tiles(emu, logn, bits):
    """Whole transforms at radix 2^4 with 4096-element row tiles, and with
    1024-element ones, the inverse also through an automorphism."""
    n = 1 << logn
    T = Tables(n, int(O.native_primes(1, bits, n)[0]))
    x = uniform(np.random.default_rng(logn + bits), T.q, n)
    for big in (0, 1):
        y = x.copy()
        emu.emu_ntt_tiles(O.P(y), n, T.q, O.P(T.fr), O.P(T.fp), 1, 0, big, 0)
        assert np.array_equal(y, T.ntt(x)), big
        for gk in (0, pow(5, 3, 2 * n), 2 * n - 1):
            y = x.copy()
            emu.emu_ntt_tiles(O.P(y), n, T.q, O.P(T.ir), O.P(T.ip), 0, int(T.ni), big, gk)
            assert np.array_equal(y, T.intt(np.ascontiguousarray(galois(x, gk)))), (big, gk)
