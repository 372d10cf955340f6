// Host emulation of the fused steps' further forms (test infrastructure, as
// emu.cpp): the inner product with a row's last step, with the tensor products
// formed there, with the dropped tower of a rescale and with digits read
// through an automorphism; the fused ModUp of up to 12 sources, the fused
// ModDown whose dropped tower is a source, and the rescale without others.
// Scratch and outputs lie between guard words; a changed one aborts.
#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <type_traits>
#include <vector>

#include "ksi.hpp"
#include "modup.hpp"
#include "ntt_engine.hpp"

using namespace gf;

namespace {
struct NoSync {
    void operator()() const {}
    void wave() const {}
};

// words between guards, 16-byte aligned
struct Guarded {
    enum : size_t { G = 64 };
    static constexpr uint64_t MARK = 0xA5A5C3C3F00D1234ull;
    std::vector<uint64_t> v;
    size_t n, at;
    explicit Guarded(size_t words) : v(words + 2 * G + 1, MARK), n(words) {
        at = G + ((uintptr_t)(v.data() + G) % 16 ? 1 : 0);
        std::fill(p(), p() + n, ~0ull);
    }
    Guarded(const Guarded&) = delete;
    uint64_t* p() { return v.data() + at; }
    ~Guarded() {
        for (size_t i = 0; i < v.size(); ++i)
            if ((i < at || i >= at + n) && v[i] != MARK) std::abort();
    }
};

std::vector<uint64_t> paired_table(const uint64_t* tw, const uint64_t* twp, uint32_t n) {
    std::vector<uint64_t> t2(2 * (size_t)n);
    for (uint32_t i = 0; i < n; ++i) {
        t2[2 * i] = tw[i];
        t2[2 * i + 1] = twp[i];
    }
    return t2;
}
std::vector<uint64_t> f64_table(const uint64_t* paired, uint32_t n, uint64_t q) {
    std::vector<uint64_t> out(2 * (size_t)n);
    for (uint32_t k = 0; k < n; ++k) {
        double wd, wq;
        f64_twiddle(paired[2 * k], q, wd, wq);
        std::memcpy(&out[2 * k], &wd, 8);
        std::memcpy(&out[2 * k + 1], &wq, 8);
    }
    return out;
}
std::vector<uint64_t> row_table(const uint64_t* paired, const NttGeom& g) {
    std::vector<uint64_t> r(row_table_words(g));
    build_row_table(paired, g, r.data());
    return r;
}

// the ring splits covered: both row lengths
template <class F>
void with_rows(const NttGeom& g, F&& f) {
    if (g.logN1 == 6 && g.logN2 == 7) f(std::integral_constant<uint32_t, 6>{}, std::integral_constant<uint32_t, 7>{});
    else if (g.logN1 == 8 && g.logN2 == 8) f(std::integral_constant<uint32_t, 8>{}, std::integral_constant<uint32_t, 8>{});
    else std::abort();
}
}  // namespace

// One row of the keyswitch's fused step.
struct KsiArgs {
    uint64_t n, q, rmax, form, np, xf, pairs, f64, gk;   // form: KSI_PLAIN, .. ; xf: transformed parts
    const uint64_t *fw, *fwp, *iw, *iwp;
    const uint64_t *src, *kb, *ka;   // [np][n]
    uint64_t *o0, *o1;               // outputs (KSI_PLAIN with drop: the inverse transforms)
    const uint64_t *v0, *v1;         // a last step's coefficient-form towers
    const uint64_t *e0, *e1;
    uint64_t ci, ce, e_plain;
    const uint64_t* in[4];
    const uint64_t *d0, *d1;         // the dropped tower's terms (with rp)
    uint64_t dpinv, post;
};

template <uint32_t RM, bool LZ, int FORM, uint32_t LOGT = KSI_LOG_TILE>
static void ksi_row(const KsiArgs& a) {
    const uint32_t n = (uint32_t)a.n;
    const uint64_t q = a.q;
    const NttGeom g = make_geom(n, RM);
    const auto ft = paired_table(a.fw, a.fwp, n), it = paired_table(a.iw, a.iwp, n);
    const auto fr = row_table(ft.data(), g), ir = row_table(it.data(), g);
    std::vector<uint64_t> ftd, itd, frd, ird;
    KsiJob J{};
    if (a.f64) {
        ftd = f64_table(ft.data(), n, q);
        itd = f64_table(it.data(), n, q);
        frd = row_table(ftd.data(), g);
        ird = row_table(itd.data(), g);
        J.twd = ftd.data();
        J.twrd = frd.data();
        J.fq = (double)q;
        J.fqinv = 1.0 / J.fq;
    }
    J.np = (uint32_t)a.np;
    J.xf = (uint32_t)a.xf;
    J.tw = ft.data();
    J.twr = fr.data();
    J.q = q;
    J.qneg = host_qneg(q);
    J.red = lazy_red_of(q);
    J.d30 = ksi_d30(q, J.red);
    J.pairs = (uint32_t)a.pairs;
    J.gk = (uint32_t)a.gk;
    J.glog = g.logn;
    // every buffer that the step reads or writes, between guards
    Guarded srcs(a.np * n), v0(n), v1(n), o0(n), o1(n);
    std::memcpy(srcs.p(), a.src, a.np * n * 8);
    J.o0 = o0.p();
    J.o1 = o1.p();
    const bool rp = a.d0 != nullptr;
    if (FORM != KSI_PLAIN) {
        std::memcpy(v0.p(), a.v0, n * 8);
        std::memcpy(v1.p(), a.v1, n * 8);
        KsiFin& F = J.fin;
        F.v[0] = v0.p();
        F.v[1] = v1.p();
        F.o[0] = o0.p();
        F.o[1] = o1.p();
        F.e[0] = a.e0;
        F.e[1] = a.e1;
        F.ci = a.ci;
        F.cip = host_precon(a.ci, q);
        F.ce = a.ce;
        F.cep = host_precon(a.ce, q);
        F.e_plain = (uint32_t)a.e_plain;
        if (FORM >= KSI_FIN_TENSOR)
            for (int k = 0; k < 4; ++k) F.in[k] = a.in[k];
        F.r2 = host_r2(q);
        if (FORM >= KSI_FIN_TENSOR && !ksi_tensor_here(J)) std::abort();
    }
    if (rp) {
        J.drop[0] = a.d0;
        J.drop[1] = a.d1;
        J.dpinv = a.dpinv;
        J.dpinvp = host_precon(a.dpinv, q);
        J.rp_on = 1;
        for (int c = 0; c < 2; ++c) {
            J.rp[c] = NttJob{nullptr, c ? o1.p() : o0.p(), it.data(), nullptr, q, a.post, host_precon(a.post, q)};
            J.rp[c].twr = ir.data();
            if (a.f64) {
                J.rp[c].twd = itd.data();
                J.rp[c].twrd = ird.data();
                J.rp[c].fq = (double)q;
                J.rp[c].fqinv = 1.0 / J.rp[c].fq;
            }
        }
    }
    with_rows(g, [&](auto A, auto B) {
        constexpr uint32_t S1 = decltype(A)::value, S2 = decltype(B)::value;
        Guarded big(NTT_TILE_PADDED);
        auto column_pass = [&](uint64_t* x) {
            NttJob t{x, x, ft.data(), nullptr, q, 0, 0};
            t.red = J.red;
            for (uint32_t tile = 0; tile < n / NTT_TILE; ++tile)
                phaseA_body<true, LZ, true, S1, RM>(t, g, tile, big.p(), 0, 1, NoSync{});
            if (a.f64)   // below 2q, as the fp64 column passes leave them
                for (uint32_t k = 0; k < n; ++k) x[k] = x[k] % q + (k % 3 == 0 ? q : 0);
        };
        for (uint32_t p = 0; p < J.np; ++p) {
            J.src[p] = srcs.p() + (size_t)p * n;
            J.kb[p] = a.kb + (size_t)p * n;
            J.ka[p] = a.ka + (size_t)p * n;
            if ((J.xf >> p) & 1) column_pass(srcs.p() + (size_t)p * n);
        }
        if (FORM != KSI_PLAIN) {
            column_pass(v0.p());
            column_pass(v1.p());
        }
        Guarded lds((size_t)ksi_regions(J) * ksi_part_words(LOGT) + (FORM == KSI_FIN_TENSOR_IN ? KSI_IN_WORDS : 0));
        for (uint32_t tile = 0; tile < n >> LOGT; ++tile) {
            std::fill(lds.p(), lds.p() + lds.n, ~0ull);   // a tile sees only what it wrote itself
            ksi_body<S2, RM, LZ, NoSync, NoSync, FORM, 6, LOGT>(J, 1u << S1, tile, lds.p(), 0, 1, 0, 1, 0, 1, NoSync{}, NoSync{});
        }
        if (rp)
            for (int c = 0; c < 2; ++c) {
                J.rp[c].twd = nullptr;   // the column pass in integers
                for (uint32_t tile = 0; tile < n / NTT_TILE; ++tile)
                    phaseA_body<false, false, true, S1, RM>(J.rp[c], g, tile, big.p(), 0, 1, NoSync{});
            }
    });
    std::memcpy(a.o0, o0.p(), n * 8);
    std::memcpy(a.o1, o1.p(), n * 8);
}

// rmax 4: the stored form on 1024-element tiles
extern "C" void emu_ksi_form(const KsiArgs* a) {
    if (a->rmax == 4) {
        if (a->form != KSI_PLAIN) std::abort();
        if (lazy_red_of(a->q)) ksi_row<4, true, KSI_PLAIN, KSI_LOG_TILE_BIG>(*a);
        else ksi_row<4, false, KSI_PLAIN, KSI_LOG_TILE_BIG>(*a);
        return;
    }
    with_row_radix((uint32_t)a->rmax, [&](auto Rc) {
        constexpr uint32_t RM = decltype(Rc)::value;
        auto form = [&](auto F) {
            constexpr int FORM = decltype(F)::value;
            if (lazy_red_of(a->q)) ksi_row<RM, true, FORM>(*a);
            else ksi_row<RM, false, FORM>(*a);
        };
        switch (a->form) {
            case KSI_PLAIN: form(std::integral_constant<int, KSI_PLAIN>{}); break;
            case KSI_FIN: form(std::integral_constant<int, KSI_FIN>{}); break;
            case KSI_FIN_TENSOR: form(std::integral_constant<int, KSI_FIN_TENSOR>{}); break;
            case KSI_FIN_TENSOR_IN: form(std::integral_constant<int, KSI_FIN_TENSOR_IN>{}); break;
        }
    });
}

// One job of the fused ModUp or ModDown, from evaluation-form sources to
// evaluation-form targets: the sources' inverse row pass, the fused kernel, the
// targets' forward row pass.  rs: the rescale mode with the dropped tower
// (q_old, its tables last) as source sp.  Targets in ranges of `len`.
struct ModupArgs {
    uint64_t n, sp, sc, rs, f64, c60, len;
    const uint64_t* const* src;                  // [sp + rs] evaluation form
    const uint64_t* sq;                          // [sp + rs]
    const uint64_t *const *sw, *const *swp;      // inverse tables
    const uint64_t* post;                        // [sp + rs]
    const uint64_t* tq;                          // [sc]
    const uint64_t *const *tw, *const *twp;      // forward tables
    const uint64_t* tab;                         // [sp][sc]
    const uint64_t* tabd;                        // [sp], rs
    uint64_t pinv;
    const uint64_t* s2;                          // [sc], rs
    uint64_t* dst;                               // [sc][n]
};

template <uint32_t SP, uint32_t S1, bool RS, bool C60>
static void modup_tiles(const ModupJob& j, const NttGeom& g) {
    Guarded lds(MODUP_TILE), tl(2u << S1);
    std::vector<uint64_t> v((size_t)MODUP_THREADS * MODUP_UNIT), dv(v.size());
    std::vector<ModupUnit<SP>> units(MODUP_THREADS);
    auto at = [](std::vector<uint64_t>& x, uint32_t u) { return x.data() + (size_t)u * MODUP_UNIT; };
    auto source = [&](uint32_t i, uint32_t tile) {
        modup_source_pass<S1, true>(j, i, g, tile, lds.p(), 0, 1, NoSync{}, v.data(), tl.p(), [&] {
            for (uint32_t k = 0; k < (1u << S1); ++k) modup_tw_put(tl.p(), k, modup_src_tw_pair(j, i, k));
        });
    };
    for (uint32_t tile = 0; tile < g.n / MODUP_TILE; ++tile) {
        for (uint32_t i = 0; i < SP; ++i) {
            source(i, tile);
            if constexpr (SP > 0)
                for (uint32_t u = 0; u < MODUP_THREADS; ++u) modup_take_unit<SP, S1>(j, i, at(v, u), units[u]);
        }
        if constexpr (RS) {
            source(SP, tile);
            for (uint32_t u = 0; u < MODUP_THREADS; ++u) modup_drop_src<SP, S1>(j, units[u], at(v, u), at(dv, u));
        }
        for (uint32_t t = j.t0; t < j.t1; ++t) {
            for (uint32_t u = 0; u < MODUP_THREADS; ++u) {
                if constexpr (RS) modup_rs_unit<SP, S1>(j, t, units[u], at(dv, u), at(v, u));
                else modup_convert_unit<SP, S1, C60>(j, t, units[u], at(v, u));
            }
            for (uint32_t i = 0; i < (1u << S1); ++i) modup_tw_put(tl.p(), i, modup_tw_pair(j, t, i));
            modup_target_pass<S1, true>(j, t, g, tile, lds.p(), 0, 1, NoSync{}, v.data(), tl.p());
        }
    }
}

extern "C" void emu_modup_form(const ModupArgs* a) {
    const uint32_t n = (uint32_t)a->n, sp = (uint32_t)a->sp, sc = (uint32_t)a->sc, ns = sp + (a->rs ? 1 : 0);
    const NttGeom g = make_geom(n, 3);
    std::vector<std::vector<uint64_t>> st(ns), sd(ns), tt(sc), td(sc);
    std::vector<uint64_t> tqn(sc), tred(sc), taddr(sc), tdaddr(sc, 0), tqf(2 * (size_t)sc), tsw(2 * (size_t)sc);
    std::vector<RsTarget> tg(sc);
    Guarded rows((size_t)ns * n), dst((size_t)sc * n), big(NTT_TILE_PADDED);
    ModupJob J{};
    with_rows(g, [&](auto A, auto B) {
        constexpr uint32_t S1 = decltype(A)::value, S2 = decltype(B)::value;
        for (uint32_t i = 0; i < ns; ++i) {
            st[i] = paired_table(a->sw[i], a->swp[i], n);
            const auto r = row_table(st[i].data(), g);
            uint64_t* x = rows.p() + (size_t)i * n;
            NttJob t{a->src[i], x, st[i].data(), nullptr, a->sq[i], 0, 0};
            t.twr = r.data();
            for (uint32_t tile = 0; tile < n / NTT_TILE; ++tile)
                phaseB_body<false, false, true, S2, 3>(t, g, tile, big.p(), 0, 1, NoSync{});
            J.src[i] = x;
            J.stw[i] = st[i].data();
            J.sq[i] = a->sq[i];
            J.post[i] = a->post[i];
            J.postp[i] = host_precon(a->post[i], a->sq[i]);
            if (a->f64 && f64_modulus(a->sq[i])) {
                sd[i] = f64_table(st[i].data(), n, a->sq[i]);
                J.stwd[i] = sd[i].data();
                J.sqd[i] = (double)a->sq[i];
                J.sqinv[i] = 1.0 / J.sqd[i];
                f64_twiddle(a->post[i], a->sq[i], J.spost[i], J.spostq[i]);
            }
        }
        const uint64_t q_old = a->rs ? a->sq[sp] : 0;
        for (uint32_t t = 0; t < sc; ++t) {
            const uint64_t q = a->tq[t];
            tt[t] = paired_table(a->tw[t], a->twp[t], n);
            tqn[t] = host_qneg(q);
            tred[t] = lazy_red_of(q);
            taddr[t] = (uint64_t)(uintptr_t)tt[t].data();
            const double qd = (double)q, qi = 1.0 / qd;
            std::memcpy(&tqf[2 * t], &qd, 8);
            std::memcpy(&tqf[2 * t + 1], &qi, 8);
            if (a->f64 && f64_modulus(q)) {
                td[t] = f64_table(tt[t].data(), n, q);
                tdaddr[t] = (uint64_t)(uintptr_t)td[t].data();
            }
            if (!a->rs) continue;
            tg[t] = RsTarget{q, tqn[t], q > q_old ? q - q_old : (q_old - q) % q, q > q_old ? 1u : 0u, a->s2[t],
                             host_precon(a->s2[t], q), host_precon(1, q)};
            rs_sw_consts(q, q_old, a->s2[t], tsw[2 * t], tsw[2 * t + 1]);
        }
        J.dst = dst.p();
        J.tab = a->tab;
        J.c60 = (uint32_t)a->c60;
        J.tq = a->tq;
        J.tqneg = tqn.data();
        J.ttw = taddr.data();
        J.tred = tred.data();
        J.ttwd = tdaddr.data();
        J.tqf = tqf.data();
        J.sp = sp;
        J.sc = sc;
        if (a->rs) {
            J.tabd = a->tabd;
            J.strided = 1;
            J.tg = tg.data();
            J.tsw = tsw.data();
            J.q_old = q_old;
            J.half = q_old >> 1;
            J.qd_neg = host_qneg(q_old);
            J.pinv = a->pinv;
            J.pinvp = host_precon(a->pinv, q_old);
        }
        auto go = [&](auto Sc) {
            constexpr uint32_t SP = decltype(Sc)::value;
            for (uint32_t t = 0; t < sc; t += (uint32_t)a->len) {
                J.t0 = t;
                J.t1 = t + (uint32_t)a->len < sc ? t + (uint32_t)a->len : sc;
                if (a->rs) modup_tiles<SP, S1, true, false>(J, g);
                else if constexpr (SP > 0) {
                    if (a->c60) {
                        if constexpr (SP <= 6) modup_tiles<SP, S1, false, true>(J, g);
                    } else {
                        modup_tiles<SP, S1, false, false>(J, g);
                    }
                }
            }
        };
#define GF_SP(k) case k: go(std::integral_constant<uint32_t, k>{}); break;
        switch (sp) {
            GF_SP(0) GF_SP(1) GF_SP(6) GF_SP(7) GF_SP(8) GF_SP(9) GF_SP(11) GF_SP(12)
            default: std::abort();
        }
#undef GF_SP
        for (uint32_t t = 0; t < sc; ++t) {
            uint64_t* y = dst.p() + (size_t)t * n;
            const auto r = row_table(tt[t].data(), g);
            NttJob k{y, y, tt[t].data(), nullptr, a->tq[t], 0, 0};
            k.twr = r.data();
            k.red = tred[t];
            for (uint32_t tile = 0; tile < n / NTT_TILE; ++tile) {
                if (k.red) phaseB_body<true, true, true, S2, 3>(k, g, tile, big.p(), 0, 1, NoSync{});
                else phaseB_body<true, false, true, S2, 3>(k, g, tile, big.p(), 0, 1, NoSync{});
            }
        }
    });
    std::memcpy(a->dst, dst.p(), (size_t)sc * n * 8);
}

// A whole transform whose row pass takes tiles of 2^12 elements at radix 2^4,
// as large launches of whole transforms do, or of 2^10 with big = 0; the inverse
// optionally reads x through the automorphism gk.
extern "C" void emu_ntt_tiles(uint64_t* x, uint64_t n, uint64_t q, const uint64_t* tw, const uint64_t* twp, int fwd,
                              uint64_t post, int big, uint64_t gk) {
    const NttGeom g = make_geom((uint32_t)n, 4);
    const auto t2 = paired_table(tw, twp, (uint32_t)n);
    const auto rows = row_table(t2.data(), g);
    Guarded in(n), out(n), lds(NTT_TILE_PADDED);
    std::memcpy(in.p(), x, n * 8);
    NttJob j{in.p(), out.p(), t2.data(), nullptr, q, post, host_precon(post, q)};
    j.twr = rows.data();
    j.red = fwd ? lazy_red_of(q) : 0;
    j.gk = (uint32_t)gk;
    j.glog = g.logn;
    with_rows(g, [&](auto A, auto B) {
        constexpr uint32_t S1 = decltype(A)::value, S2 = decltype(B)::value;
        auto rows_of = [&](auto L, auto T, auto F) {
            constexpr uint32_t LOGT = decltype(T)::value;
            for (uint32_t t = 0; t < n >> LOGT; ++t)
                phaseB_body<decltype(F)::value, decltype(L)::value, true, S2, 4, NoSync, false, LOGT>(j, g, t, lds.p(), 0, 1, NoSync{});
        };
        auto cols_of = [&](auto L, auto F) {
            for (uint32_t t = 0; t < n >> NTT_LOG_TILE_BIG; ++t)
                phaseA_body<decltype(F)::value, decltype(L)::value, true, S1, 4, NoSync, NTT_LOG_TILE_BIG>(j, g, t, lds.p(), 0, 1, NoSync{});
        };
        using Small = std::integral_constant<uint32_t, NTT_LOG_TILE>;
        using Big = std::integral_constant<uint32_t, NTT_LOG_TILE_BIG>;
        auto run_rows = [&](auto L, auto F) {
            if (big) rows_of(L, Big{}, F);
            else rows_of(L, Small{}, F);
        };
        if (!fwd) {
            run_rows(std::false_type{}, std::false_type{});
            cols_of(std::false_type{}, std::false_type{});
        } else if (j.red) {
            cols_of(std::true_type{}, std::true_type{});
            run_rows(std::true_type{}, std::true_type{});
        } else {
            cols_of(std::false_type{}, std::true_type{});
            run_rows(std::false_type{}, std::true_type{});
        }
    });
    std::memcpy(x, out.p(), n * 8);
}
