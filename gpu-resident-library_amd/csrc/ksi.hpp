// Fused last pass of the ModUp digits' forward transform and the key inner
// product (the inner product of src/keyswitch_resident.cpp:171-200 over
// digits produced by the forward NTT of :184-194).
//
// One workgroup owns KSI_TILE consecutive positions of tower row i (ROWS
// transform rows of N2) for every part p of the decomposition.  Wave w runs
// the forward row pass (phase B) of the transformed parts w, w + nwaves, ...
// (in part order) on LDS region w, w + nwaves, ..., reading the phase-A output
// straight from HBM, and keeps the evaluation-form digits there; after one
// block barrier every thread (including an optional extra wave that runs no
// row pass) takes KSI_TILE / nthr positions and accumulates
// sum_p digit_p * key_p for both key components (30-bit column sums where
// every value is below 2^60 and there are at most 6 parts, else 128-bit sums).  A launch
// gives its jobs one wave per transformed part (up to KSI_WAVES), so no wave
// idles through the row passes.  The transformed digits therefore never
// travel through HBM.  Parts whose tower i is the input's own (no transform)
// are read from HBM at the inner product.
#pragma once
#include "ntt_engine.hpp"
#include "ntt_f64.hpp"
#include "tensor.hpp"

namespace gf {

// Tiles of 512 positions: one radix-8 unit per lane and pass, half the LDS
// and half the serial work per workgroup of 1024.  The row passes wait on
// memory and the inner product on memory, so what counts is how many
// workgroups a CU holds and how evenly they interleave (64 EvalMult+Rescale at
// n = 2^16, L = 24: 7690 -> 7590 us; a 10-deep chain of 16 at n = 2^15: 3418 ->
// 3231; one rotation at n = 2^15: 115 -> 98).  256 positions leave half the
// lanes of a pass idle (8490 us).  Large launches over integer rows of 256 words
// take 1024 where the tuner chose radix 2^4: a unit of 16 per lane, and two passes
// instead of three (Ctx::big_ksi_tiles).
enum {
    KSI_MAXP = 7,                                    // parts per job (KSI_MAXP regions fit 64 KiB of LDS)
    KSI_LOG_TILE = 9,
    KSI_TILE = 1 << KSI_LOG_TILE,                    // positions per workgroup
    KSI_PART_WORDS = KSI_TILE + KSI_TILE / 16,       // one part's padded LDS region
    KSI_LOG_TILE_BIG = 10,                           // (Ctx::big_ksi_tiles)
    KSI_WAVES = 7,                                   // largest workgroup, in waves
    KSI_THREADS = 64 * KSI_WAVES
};

GF_HD constexpr uint32_t ksi_part_words(uint32_t logt) { return (1u << logt) + (1u << logt) / 16; }

// The last step of an output row of both components c, in the launch that
// forms its inner products r_c: v[c] is the column-pass output of the ModDown's
// forward transform; its row pass runs beside the digits' (two more LDS
// regions, after the parts'), and the row is stored as
//   o[c] = NTT(v[c]) + r_c ci + e[c] (times ce unless e_plain; e[c] may be null
//   with e_plain)
// so the inner products never travel through HBM.
struct KsiFin {
    const uint64_t* v[2];
    uint64_t* o[2];
    const uint64_t* e[2];
    uint64_t ci, cip, ce, cep;
    uint32_t e_plain;
    // in[0] set (ksi_tensor_here): the two ciphertexts' rows c0a, c1a, c0b, c1b.
    // e[0], e[1] and the untransformed digit are their tensor products, formed
    // here and not read: the row's three products are not stored and read
    // again for the price of one more input row.
    const uint64_t* in[4];
    uint64_t r2;   // 2^128 mod q
};

struct KsiJob {
    // part p's tower of row i: the phase-A output of its forward transform
    // (bit p of xf set) or an evaluation-form digit read as it is
    const uint64_t* src[KSI_MAXP];
    const uint64_t* kb[KSI_MAXP];   // key rows (Montgomery form)
    const uint64_t* ka[KSI_MAXP];
    uint64_t* o0;
    uint64_t* o1;
    const uint64_t* tw;     // paired forward twiddles of row i's modulus
    const uint64_t* twr;    // and their phase-B row table
    uint64_t q, qneg;
    uint64_t red;           // lazy_red_of(q): the transforms skip their reductions
    uint32_t np, xf;
    uint32_t pairs;         // every tower pointer 16-byte aligned: two positions per access
    // 1: the outputs only feed the rescale epilogue's lazy Shoup products
    // (any 64-bit input): REDC without its correction, no final reduction
    uint32_t lazy_out;
    // 1: every digit and key value of the row is below 2^60 (ksi_d30), so the
    // inner product runs as 30-bit column sums
    uint32_t d30;
    // digits from the fp64 ModUp (below 2q) of a modulus below 2^50: the row
    // passes in fp64 (ntt_f64.hpp) with these pairs and their row table, q and
    // fl(1/q); null: the integer passes
    const uint64_t* twd;
    const uint64_t* twrd;
    double fq, fqinv;
    // rp_on: the row's two outputs are not stored; instead the inverse
    // transforms' row pass rp[c] (its input tower o0 / o1) runs on them after
    // the inner product, from LDS (two LDS regions at least, ksi_regions)
    uint32_t rp_on;
    NttJob rp[2];
    // with rp_on, the dropped tower of a rescale (else null): the row pass runs
    // on drop[c] + output times dpinv (dpinv = P^-1 mod q), the evaluation form
    // of the dropped tower but for its ModDown conversion
    const uint64_t* drop[2];
    uint64_t dpinv, dpinvp;
    // parts that are not transformed here (and fin.e with fin.e_plain) are read
    // through the automorphism of index gk (0: as they are), n = 2^glog
    uint32_t gk, glog;
    // fin.v[0] set: the row's last step (KsiFin) instead of o0, o1
    KsiFin fin;
};
// LDS regions of a job: one per transformed part, two at least where the row
// pass takes its outputs, and two more for a last step's row passes
inline uint32_t ksi_regions(const KsiJob& j) {
    const uint32_t x = (uint32_t)__builtin_popcount(j.xf);
    return j.fin.v[0] ? x + 2 : j.rp_on && x < 2 ? 2 : x;
}

// V consecutive words from word i of a tower (V = 2: one 16-byte access; the
// address is 16-byte aligned), addressed as base + 32-bit byte offset (gat)
template <uint32_t V>
GF_HD void load_words(const GF_GLOBAL uint64_t* base, uint32_t i, uint64_t* out) {
    if constexpr (V == 2) {
        const Words2 x = gat((const GF_GLOBAL Words2*)base, i / 2);
        out[0] = x.w[0];
        out[1] = x.w[1];
    } else {
        out[0] = gat(base, i);
    }
}
template <uint32_t V>
GF_HD void store_words(GF_GLOBAL uint64_t* base, uint32_t i, const uint64_t* in) {
    if constexpr (V == 2) {
        gat((GF_GLOBAL Words2*)base, i / 2) = Words2{{in[0], in[1]}};
    } else {
        gat(base, i) = in[0];
    }
}

// the same at position i of the automorphism gk's image (V = 2: i even; see
// galois_index)
template <uint32_t V>
GF_HD void load_words_gk(const GF_GLOBAL uint64_t* base, uint32_t i, uint32_t gk, uint32_t glog, uint64_t* out) {
    const uint32_t g = galois_index(i, gk, glog);
    if constexpr (V == 2) {
        const Words2 x = gat((const GF_GLOBAL Words2*)base, g / 2);
        out[0] = g & 1 ? x.w[1] : x.w[0];
        out[1] = g & 1 ? x.w[0] : x.w[1];
    } else {
        out[0] = gat(base, g);
    }
}
template <uint32_t V>
GF_HD void load_words_any(const GF_GLOBAL uint64_t* base, uint32_t i, const KsiJob& j, uint64_t* out) {
    if (j.gk) load_words_gk<V>(base, i, j.gk, j.glog, out);
    else load_words<V>(base, i, out);
}

// Digits and keys of a row fit the 30-bit column sums when both are below
// 2^60: keys are residues (< q); digits are residues too, or with red (the
// forward transform's unreduced values) below 72 q.
inline uint32_t ksi_d30(uint64_t q, uint64_t red) {
    const unsigned __int128 dmax = red ? (unsigned __int128)72 * q : (unsigned __int128)q;
    return dmax <= ((unsigned __int128)1 << 60) ? 1u : 0u;
}

// The inner product's outputs at positions idx .. idx + V - 1 (word gi of the
// row): to HBM, or (j.rp_on) into LDS regions 0 and 1 at those positions'
// slots for the row pass after it; each thread writes only its own
// positions, whose digits it has already read
// the forms of the kernel: inner products stored (or through rp), with the
// rows' last step, and with the tensor products formed there
// KSI_FIN_TENSOR_IN: KSI_FIN_TENSOR with the input towers' tile through LDS
// (ksi_request_inputs), a launch's choice (run_ksi)
enum { KSI_PLAIN = 0, KSI_FIN = 1, KSI_FIN_TENSOR = 2, KSI_FIN_TENSOR_IN = 3 };

// the jobs whose last step may form the tensor products itself: the column
// sums' form of the inner product with two positions per access
inline bool ksi_tensor_here(const KsiJob& j) { return j.fin.v[0] && j.d30 && j.np <= 6 && j.pairs; }

// The tensor products of one position: t0, t1 for the lazy Shoup products and
// t2 as a digit below 2^60.  fp64 rows: exact products in (-q, q) each, shifted
// into [0, 4q).
GF_HD void ksi_tensor(const KsiJob& j, const uint64_t* x, uint64_t& t0, uint64_t& t1, uint64_t& t2) {
    if (j.twd) {
        const double q = j.fq, qi = j.fqinv;
        const double a0 = f64_from_u52(x[0], F64_2P52), a1 = f64_from_u52(x[1], F64_2P52),
                     b0 = f64_from_u52(x[2], F64_2P52), b1 = f64_from_u52(x[3], F64_2P52);
        t0 = u52_from_f64(f64_mulres(a0, b0, q, qi) + q);
        t1 = u52_from_f64(f64_mulres(a0, b1, q, qi) + f64_mulres(a1, b0, q, qi) + 2 * q);
        t2 = u52_from_f64(f64_mulres(a1, b1, q, qi) + q);
        return;
    }
    TensorJob t{};
    t.q = j.q;
    t.qneg = j.qneg;
    t.r2 = j.fin.r2;
    tensor_one(t, x[0], x[1], x[2], x[3], t0, t1, t2);
}

// The four input towers' tile of a last step that forms the tensor products
// goes to LDS behind the job's regions, straight from HBM, requested before the
// row passes: one round trip to HBM less behind the barrier, and no registers
// held for it.
enum { KSI_IN_WORDS = 4 * KSI_TILE, KSI_IN_CHUNK = 128 };   // a chunk: one 16-byte access per lane
GF_HD uint32_t ksi_in_off(const KsiJob& j) { return ((uint32_t)__builtin_popcount(j.xf) + 2) * KSI_PART_WORDS; }
GF_HD void ksi_request_inputs(const KsiJob& j, uint64_t* lds, uint32_t off, uint32_t wave, uint32_t nwaves,
                              uint32_t lane, uint32_t wlanes) {
#if defined(__HIP_DEVICE_COMPILE__)
    for (uint32_t c = __builtin_amdgcn_readfirstlane(wave); c < KSI_IN_WORDS / KSI_IN_CHUNK; c += nwaves) {
        const uint32_t k = c / (KSI_TILE / KSI_IN_CHUNK), o = c % (KSI_TILE / KSI_IN_CHUNK) * KSI_IN_CHUNK;
        const GF_GLOBAL uint64_t* src = gcast(j.fin.in[k]) + off + o + 2 * lane;
        __builtin_amdgcn_global_load_lds((const GF_GLOBAL void*)src,
                                         (__attribute__((address_space(3))) void*)(lds + ksi_in_off(j) + c * KSI_IN_CHUNK),
                                         16, 0, 0);
    }
#else
    for (uint32_t i = wave * wlanes + lane; i < KSI_IN_WORDS; i += nwaves * wlanes)
        lds[ksi_in_off(j) + i] = j.fin.in[i / KSI_TILE][off + i % KSI_TILE];
#endif
}
// this wave's requests have arrived (the workgroup barrier follows)
GF_HD void ksi_wait_inputs() {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#endif
}

template <uint32_t V>
struct KsiEps {
    uint64_t e0[V], e1[V];   // fin.e[c] at the step's positions
};
// the last step's operands, requested with the step's other loads
template <int FIN, uint32_t V>
GF_HD void ksi_load_eps(const KsiJob& j, uint32_t gi, KsiEps<V>& x) {
    if constexpr (FIN == KSI_FIN) {
        if (j.fin.e_plain) {
            if (j.fin.e[0]) load_words_any<V>(gcast(j.fin.e[0]), gi, j, x.e0);
            if (j.fin.e[1]) load_words_any<V>(gcast(j.fin.e[1]), gi, j, x.e1);
        } else {
            load_words<V>(gcast(j.fin.e[0]), gi, x.e0);
            load_words<V>(gcast(j.fin.e[1]), gi, x.e1);
        }
    }
}
template <int FIN, bool LZ, uint32_t V, uint32_t PART>
GF_HD void ksi_store(const KsiJob& j, uint64_t* lds, uint32_t idx, uint32_t gi, const uint64_t* r0,
                     const uint64_t* r1, const KsiEps<V>& x, const NttJob& t) {
    if constexpr (FIN) {
        const uint32_t k0 = (uint32_t)__builtin_popcount(j.xf) * PART;
        auto comp = [&](uint32_t c, const uint64_t* r, const uint64_t* e) {
            uint64_t y[V];
            const int ep = FIN >= KSI_FIN_TENSOR || !j.fin.e_plain ? 0 : j.fin.e[c] ? 1 : 2;
#pragma unroll
            for (uint32_t v = 0; v < V; ++v) {
                const uint64_t z = lds[k0 + c * PART + padded(idx + v)];
                y[v] = ep == 0   ? ntt_ep_value<LZ, 0>(z, t, r[v], e[v])
                       : ep == 1 ? ntt_ep_value<LZ, 1>(z, t, r[v], e[v])
                                 : ntt_ep_value<LZ, 2>(z, t, r[v], 0);
            }
            store_words<V>(gcast(j.fin.o[c]), gi, y);
        };
        comp(0, r0, x.e0);
        comp(1, r1, x.e1);
        return;
    }
    if (j.rp_on) {
        uint64_t t0[V], t1[V];
        if (j.drop[0]) {
            load_words<V>(gcast(j.drop[0]), gi, t0);
            load_words<V>(gcast(j.drop[1]), gi, t1);
        }
#pragma unroll
        for (uint32_t v = 0; v < V; ++v) {
            uint64_t a = r0[v], b = r1[v];
            if (j.drop[0]) {
                a = addmod(t0[v], shoup(a, j.dpinv, j.dpinvp, j.q), j.q);
                b = addmod(t1[v], shoup(b, j.dpinv, j.dpinvp, j.q), j.q);
            }
            lds[padded(idx + v)] = a;
            lds[PART + padded(idx + v)] = b;
        }
        return;
    }
    store_words<V>(gcast(j.o0), gi, r0);
    store_words<V>(gcast(j.o1), gi, r1);
}

// hi:lo of lo + mid 2^30 + hi 2^60 (the column sums of dot30's layout)
GF_HD U128 cols_to_u128(uint64_t lo, uint64_t mid, uint64_t hi) {
    U128 T;
    T.lo = lo + (mid << 30);
    uint64_t c = T.lo < lo ? 1u : 0u;
    const uint64_t h = hi << 60;
    T.lo += h;
    c += T.lo < h ? 1u : 0u;
    T.hi = (mid >> 34) + (hi >> 4) + c;
    return T;
}

// The inner product of NP parts (NP known at compile time): positions
// idx .. idx + V - 1 per step; all operands of a step (each part's digit, from
// LDS or HBM, and both key rows) are loaded before any arithmetic, and the
// sums are 30-bit column sums (j.d30): per part and component four 32 x 32
// multiply-adds with no carries.  NP <= 7 keeps every column below 2^64
// (lo, hi < 7 2^60; mid < 14 2^60).
template <uint32_t NP, uint32_t V, bool LZ, int FIN, uint32_t LOGT>
GF_HD void ksi_inner_cols(const KsiJob& j, uint64_t* lds, uint32_t off, uint32_t tid, uint32_t nthr,
                          const NttJob& t) {
    const GF_GLOBAL uint64_t *src[NP], *kb[NP], *ka[NP];
    uint32_t reg[NP];
    bool xf[NP];
#pragma unroll
    for (uint32_t p = 0; p < NP; ++p) {
        src[p] = gcast(j.src[p]);
        kb[p] = gcast(j.kb[p]);
        ka[p] = gcast(j.ka[p]);
        xf[p] = (j.xf >> p) & 1;
        reg[p] = (uint32_t)__builtin_popcount(j.xf & ((1u << p) - 1)) * ksi_part_words(LOGT);
    }
    const uint64_t q = j.q, qneg = j.qneg;
    for (uint32_t idx = tid * V; idx < 1u << LOGT; idx += nthr * V) {
        const uint32_t gi = off + idx;
        uint64_t dv[NP][V], bv[NP][V], av[NP][V];
#pragma unroll
        for (uint32_t p = 0; p < NP; ++p) {
            if (xf[p]) {
#pragma unroll
                for (uint32_t v = 0; v < V; ++v) dv[p][v] = lds[reg[p] + padded(idx + v)];
            } else if constexpr (FIN < KSI_FIN_TENSOR) {
                load_words_any<V>(src[p], gi, j, dv[p]);
            }
            load_words<V>(kb[p], gi, bv[p]);
            load_words<V>(ka[p], gi, av[p]);
        }
        KsiEps<V> ep;
        ksi_load_eps<FIN, V>(j, gi, ep);
        if constexpr (FIN >= KSI_FIN_TENSOR) {
            uint64_t x[4][V];
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) {
                if constexpr (FIN == KSI_FIN_TENSOR_IN) {
#pragma unroll
                    for (uint32_t v = 0; v < V; ++v) x[k][v] = lds[ksi_in_off(j) + k * KSI_TILE + idx + v];
                } else {
                    load_words<V>(gcast(j.fin.in[k]), gi, x[k]);
                }
            }
#pragma unroll
            for (uint32_t v = 0; v < V; ++v) {
                const uint64_t y[4] = {x[0][v], x[1][v], x[2][v], x[3][v]};
                uint64_t t2;
                ksi_tensor(j, y, ep.e0[v], ep.e1[v], t2);
#pragma unroll
                for (uint32_t p = 0; p < NP; ++p)
                    if (!xf[p]) dv[p][v] = t2;
            }
        }
        uint64_t r0[V], r1[V];
#pragma unroll
        for (uint32_t v = 0; v < V; ++v) {
            uint64_t l0 = 0, m0 = 0, h0 = 0, l1 = 0, m1 = 0, h1 = 0;
#pragma unroll
            for (uint32_t p = 0; p < NP; ++p) {
                uint64_t d = dv[p][v];
                // LZ: below 72q < 2^60 as is (j.d30); else [0, 8q) -> [0, q)
                if (!LZ && xf[p]) d = ntt_final<true>(d, t);
                const uint32_t d0 = split30_lo(d), d1 = split30_hi(d);
                const uint64_t b = bv[p][v], a = av[p][v];
                const uint32_t b0 = split30_lo(b), b1 = split30_hi(b), a0 = split30_lo(a), a1 = split30_hi(a);
                l0 = mad32(d0, b0, l0);
                m0 = mad32(d0, b1, m0);
                m0 = mad32(d1, b0, m0);
                h0 = mad32(d1, b1, h0);
                l1 = mad32(d0, a0, l1);
                m1 = mad32(d0, a1, m1);
                m1 = mad32(d1, a0, m1);
                h1 = mad32(d1, a1, h1);
            }
            const U128 s0 = cols_to_u128(l0, m0, h0), s1 = cols_to_u128(l1, m1, h1);
            if (FIN || j.lazy_out) {
                r0[v] = redc_lazy(s0, q, qneg);
                r1[v] = redc_lazy(s1, q, qneg);
            } else if constexpr (LZ) {
                r0[v] = redc_red(s0, q, qneg, (uint32_t)j.red);
                r1[v] = redc_red(s1, q, qneg, (uint32_t)j.red);
            } else {
                r0[v] = redc(s0, q, qneg);
                r1[v] = redc(s1, q, qneg);
            }
        }
        ksi_store<FIN, LZ, V, ksi_part_words(LOGT)>(j, lds, idx, gi, r0, r1, ep, t);
    }
}

// ksi_inner_cols for the job's part count, when it has an instantiation
template <uint32_t V, bool LZ, int FIN, int NPMAX, uint32_t LOGT>
GF_HD bool ksi_inner_cols_np(const KsiJob& j, uint64_t* lds, uint32_t off, uint32_t tid, uint32_t nthr,
                             const NttJob& t) {
    switch (j.np) {
        case 1: ksi_inner_cols<1, V, LZ, FIN, LOGT>(j, lds, off, tid, nthr, t); return true;
        case 2: ksi_inner_cols<2, V, LZ, FIN, LOGT>(j, lds, off, tid, nthr, t); return true;
        case 3: ksi_inner_cols<3, V, LZ, FIN, LOGT>(j, lds, off, tid, nthr, t); return true;
        case 4: ksi_inner_cols<4, V, LZ, FIN, LOGT>(j, lds, off, tid, nthr, t); return true;
        // 5 and 6 parts take one position per access (two need more registers
        // than 5 waves per SIMD leave).  Beside the other counts their operands'
        // scalar loads spill SGPRs (42 to 49 in the plain form, 213 to 255 with the
        // last step, 49 to 68 with the tensor products), so only launches that have
        // such jobs take a kernel with all six (NPMAX = 6; 59 EvalMult+Rescale of
        // 19 towers in 5 parts at n = 2^14: 1580 us by 128-bit sums, 1503 by these);
        // the other launches' kernels spill none, 33 to 41, and up to 6.
        case 5:
            if constexpr (NPMAX >= 5) {
                ksi_inner_cols<5, 1, LZ, FIN, LOGT>(j, lds, off, tid, nthr, t);
                return true;
            }
            return false;
        case 6:
            if constexpr (NPMAX >= 6) {
                ksi_inner_cols<6, 1, LZ, FIN, LOGT>(j, lds, off, tid, nthr, t);
                return true;
            }
            return false;
        default: return false;
    }
}

// LZ = (j.red != 0), FIN = KSI_FIN where j.fin.v[0] is set, KSI_FIN_TENSOR
// where j.fin.in[0] is too, else KSI_PLAIN.  The wave-level sync wsync separates the row passes of
// one wave's region; bsync is the workgroup barrier before the inner product.
template <uint32_t S2, uint32_t RM, bool LZ, class WSync, class BSync, int FIN = KSI_PLAIN, int NPMAX = 4,
          uint32_t LOGT = KSI_LOG_TILE>
GF_HD void ksi_body(const KsiJob& j, uint32_t N1, uint32_t tile, uint64_t* lds, uint32_t wave, uint32_t nwaves,
                    uint32_t lane, uint32_t wlanes, uint32_t tid, uint32_t nthr, WSync wsync, BSync bsync) {
    constexpr uint32_t ROWS = (1u << LOGT) >> S2, LOGR = LOGT - S2, PART = ksi_part_words(LOGT);
    const uint32_t a0 = tile * ROWS, off = a0 << S2;
    NttJob t{};
    t.tw = j.tw;
    t.twr = j.twr;
    t.q = j.q;
    t.red = j.red;
    const TileDesc d{LOGR, 1, padded(1u << S2), N1 + a0, 1, false, true};
    // transformed part k (in part order) -> LDS region k, then a last step's
    // two components
    uint32_t k = 0;
    auto row_pass = [&](const uint64_t* src) {
        if (k % nwaves == wave) {
            if (j.twd)
                row_tile_f64<true, S2, RM, ROWS, true>(j.twd, j.twrd, j.fq, j.fqinv, d, gcast(src), nullptr, off,
                                                       lds + k * PART, lane, wlanes, wsync);
            else
                row_tile<true, LZ, true, S2, RM, ROWS, 2, true, WSync, true>(
                    t, d, gcast(src), nullptr, off, lds + k * PART, lane, wlanes, wsync);
        }
        ++k;
    };
    const uint32_t np = j.np, rows = FIN ? np + 2 : np;
    if constexpr (FIN == KSI_FIN_TENSOR_IN) ksi_request_inputs(j, lds, off, wave, nwaves, lane, wlanes);
    for (uint32_t p = 0; p < rows; ++p) {
        if (p < np) {
            if ((j.xf >> p) & 1) row_pass(j.src[p]);
        } else {
            row_pass(j.fin.v[p - np]);
        }
    }
    if constexpr (FIN) {
        // the last step as a forward transform's epilogue (ntt_ep_value)
        t.c0 = j.fin.ci;
        t.c0p = j.fin.cip;
        t.c1 = j.fin.ce;
        t.c1p = j.fin.cep;
    }
    if constexpr (FIN == KSI_FIN_TENSOR_IN) ksi_wait_inputs();
    bsync();
    // up to 6 parts with every value below 2^60: column sums, loads first
    bool done = false;
    if (j.d30)
        done = FIN >= KSI_FIN_TENSOR || j.pairs ? ksi_inner_cols_np<2, LZ, FIN, NPMAX, LOGT>(j, lds, off, tid, nthr, t)
                                                : ksi_inner_cols_np<1, LZ, FIN, NPMAX, LOGT>(j, lds, off, tid, nthr, t);
    // positions idx .. idx + V - 1 per step (V = 2: one 16-byte access per operand)
    auto inner = [&](auto Vc) {
        constexpr uint32_t V = decltype(Vc)::value;
        const uint64_t q = j.q, qneg = j.qneg;
        for (uint32_t idx = tid * V; idx < 1u << LOGT; idx += nthr * V) {
            const uint32_t gi = off + idx;
            U128 s0[V], s1[V];
            for (uint32_t v = 0; v < V; ++v) s0[v] = s1[v] = U128{0, 0};
            for (uint32_t p = 0; p < j.np; ++p) {
                uint64_t dv[V], kb[V], ka[V];
                if ((j.xf >> p) & 1) {
                    const uint32_t k = __builtin_popcount(j.xf & ((1u << p) - 1));
                    for (uint32_t v = 0; v < V; ++v) {
                        dv[v] = lds[k * PART + padded(idx + v)];
                        // LZ: below 72q (the sums stay below 2^125); else [0, 8q) -> [0, q)
                        if constexpr (!LZ) dv[v] = ntt_final<true>(dv[v], t);
                    }
                } else {
                    load_words_any<V>(gcast(j.src[p]), gi, j, dv);
                }
                load_words<V>(gcast(j.kb[p]), gi, kb);
                load_words<V>(gcast(j.ka[p]), gi, ka);
                for (uint32_t v = 0; v < V; ++v) {
                    s0[v] = add128(s0[v], mul128(dv[v], kb[v]));
                    s1[v] = add128(s1[v], mul128(dv[v], ka[v]));
                }
            }
            uint64_t r0[V], r1[V];
            for (uint32_t v = 0; v < V; ++v) {
                if (FIN || j.lazy_out) {
                    r0[v] = redc_lazy(s0[v], q, qneg);
                    r1[v] = redc_lazy(s1[v], q, qneg);
                } else if constexpr (LZ) {
                    r0[v] = redc_red(s0[v], q, qneg, (uint32_t)j.red);
                    r1[v] = redc_red(s1[v], q, qneg, (uint32_t)j.red);
                } else {
                    r0[v] = redc(s0[v], q, qneg);
                    r1[v] = redc(s1[v], q, qneg);
                }
            }
            KsiEps<V> ep;
            ksi_load_eps<FIN, V>(j, gi, ep);
            ksi_store<FIN, LZ, V, PART>(j, lds, idx, gi, r0, r1, ep, t);
        }
    };
    if (FIN < KSI_FIN_TENSOR && !done) {   // (those jobs have the column sums' form)
        if (j.pairs) inner(std::integral_constant<uint32_t, 2>{});
        else inner(std::integral_constant<uint32_t, 1>{});
    }
    // the inverse transforms' row pass of the two output rows (inputs in
    // [0, q), lazy outputs for the column pass after it), component c by
    // wave c
    if (!FIN && j.rp_on) {
        bsync();
        for (uint32_t c = wave; c < 2; c += nwaves) {
            const NttJob& r = j.rp[c];
            if (r.twd)
                row_tile_f64<false, S2, RM, ROWS, false, WSync, true>(r.twd, r.twrd, r.fq, r.fqinv, d, nullptr,
                                                                      gcast(r.out), off, lds + c * PART, lane,
                                                                      wlanes, wsync);
            else
                row_tile<false, false, true, S2, RM, ROWS, 0, true, WSync, false, true>(
                    r, d, nullptr, gcast(r.out), off, lds + c * PART, lane, wlanes, wsync);
        }
    }
}

}  // namespace gf
