// The fused ModUp kernel (modup.hpp), shared by the translation units that
// instantiate it: kernels_modup.hip (up to 6 sources), kernels_modup_w.hip and
// kernels_moddown_w.hip (7 to 12), apart so that they compile in parallel.
#pragma once
#include "modup.hpp"
#include "ntt_kernels.hpp"

namespace gf {

// One workgroup per (part job, column tile).  Source count SP fixed at compile
// time, so every thread's unit of the sources stays in registers.
// Sources I .. SP - 1, one after the other (compile-time source index, so the
// unit arrays are indexed by constants and stay in registers); source I is
// phase I and takes LDS tile I mod 2 and twiddle tile I mod 2; its twiddles
// are requested with its first pass's data
// source i's inverse column pass into the unit registers v, as phase i
template <uint32_t S1>
__device__ __forceinline__ void modup_source(const ModupJob& j, uint32_t i, const NttGeom& g, uint64_t* lds,
                                             uint64_t (*twl)[2u << S1], uint32_t tid, uint32_t tile, uint64_t* v) {
    constexpr uint32_t TWP = 1u << S1, TWPER = TWP > MODUP_THREADS ? TWP / MODUP_THREADS : 1;
    Words2 tp[TWPER];
#pragma unroll
    for (uint32_t k = 0; k < TWPER; ++k)
        if (tid + k * MODUP_THREADS < TWP) tp[k] = modup_src_tw_pair(j, i, tid + k * MODUP_THREADS);
    uint64_t* tl = twl[i & 1];
    modup_source_pass<S1, false>(j, i, g, tile, lds + (i & 1) * MODUP_TILE, tid, MODUP_THREADS, DevSync{}, v, tl, [&] {
#pragma unroll
        for (uint32_t k = 0; k < TWPER; ++k)
            if (tid + k * MODUP_THREADS < TWP) modup_tw_put(tl, tid + k * MODUP_THREADS, tp[k]);
    });
}
template <uint32_t S1, uint32_t SP, uint32_t I>
__device__ __forceinline__ void modup_sources(const ModupJob& j, const NttGeom& g, uint64_t* lds,
                                              uint64_t (*twl)[2u << S1], uint32_t tid, uint32_t tile,
                                              ModupUnit<SP>& x) {
    if constexpr (I < SP) {
        uint64_t v[MODUP_UNIT];
        modup_source<S1>(j, I, g, lds, twl, tid, tile, v);
        modup_take_unit<SP, S1>(j, I, v, x);
        modup_sources<S1, SP, I + 1>(j, g, lds, twl, tid, tile, x);
    }
}

// One workgroup's tile of a job with SP sources.  RS: the rescale mode (the
// fused ModDown + rescale prologue; ModupJob); C60: the conversion's R = 2^60
// column reduction (ModupJob::c60).
template <uint32_t S1, uint32_t SP, bool RS, bool C60>
__device__ __forceinline__ void modup_run(const ModupJob& j, const NttGeom& g, uint64_t* lds,
                                          uint64_t (*twl)[2u << S1], uint32_t tid, uint32_t tile) {
    constexpr uint32_t TWP = 1u << S1, TWPER = TWP > MODUP_THREADS ? TWP / MODUP_THREADS : 1;
    ModupUnit<SP> x;
    modup_sources<S1, SP, 0>(j, g, lds, twl, tid, tile, x);
    // target t is phase ph0 + t - t0; its twiddles are requested before its
    // conversion and stored to LDS after it
    uint64_t cv[MODUP_UNIT];
    const uint32_t t0 = j.t0, t1 = j.t1, ph0 = SP + (RS && j.src[SP] ? 1 : 0);
    auto target = [&](uint32_t t, auto&& convert) {
        Words2 tp[TWPER];
#pragma unroll
        for (uint32_t k = 0; k < TWPER; ++k)
            if (tid + k * MODUP_THREADS < TWP) tp[k] = modup_tw_pair(j, t, tid + k * MODUP_THREADS);
        convert();
        const uint32_t ph = (ph0 + t - t0) & 1;
        uint64_t* tl = twl[ph];
#pragma unroll
        for (uint32_t k = 0; k < TWPER; ++k)
            if (tid + k * MODUP_THREADS < TWP) modup_tw_put(tl, tid + k * MODUP_THREADS, tp[k]);
        modup_target_pass<S1, false>(j, t, g, tile, lds + ph * MODUP_TILE, tid, MODUP_THREADS, DevSync{}, cv, tl);
    };
    if constexpr (RS) {
        uint64_t dv[MODUP_UNIT];
        if (j.src[SP]) {
            modup_source<S1>(j, SP, g, lds, twl, tid, tile, cv);
            modup_drop_src<SP, S1>(j, x, cv, dv);
        } else if constexpr (SP > 0) {
            modup_drop_unit<SP, S1>(j, g, tile, tid, x, dv);
        }
        for (uint32_t t = t0; t < t1; ++t) target(t, [&] { modup_rs_unit<SP, S1>(j, t, x, dv, cv); });
    } else {
        for (uint32_t t = t0; t < t1; ++t) target(t, [&] { modup_convert_unit<SP, S1, C60>(j, t, x, cv); });
    }
}

// The jobs of one launch have up to SPMAX sources each; the branch on a job's
// count is uniform per workgroup.  One launch for every source count: a batch
// of uneven levels has a few jobs of each count below the part width, and
// launched apart those launches fill a part of the chip each (rotations of 64
// ciphertexts at levels 8..20, n = 2^16: five launches of 63, 68, 81, 89 and
// 744 us became one of 898).  SPMAX keeps the registers of small
// contexts down (8 per source); jobs of 7 to 12 sources (SPMAX = 12) have 168
// registers and 3 waves per SIMD, in launches of their own, and at 12 sources
// still spill some (ModUp 14 to 54 registers by ring split, 54 at n = 2^16; ModDown
// 2 to 19): 8 EvalMult+Rescale at n = 2^16, L = 24, dnum = 2 run 963 us with them,
// 1367 unfused; one of 17 towers at n = 2^14, dnum = 2 103 us, 171 unfused.
template <uint32_t S1, uint32_t SPMAX, bool RS, bool C60>
__global__ __launch_bounds__(MODUP_THREADS) __attribute__((amdgpu_waves_per_eu(SPMAX > 6 ? 3 : 4, 8))) void k_modup(const ModupJob* __restrict__ jobs, uint32_t off, NttGeom g) {
    __shared__ uint64_t lds[2 * MODUP_TILE];   // phases alternate between the two tiles
    // the phases' column-pass twiddles (modup_src_tw_pair, modup_tw_pair), by
    // phase parity as the tiles: phase p + 2 rewrites phase p's copy only
    // after a barrier of phase p + 1, which every thread reaches after its
    // last read of it
    __shared__ uint64_t twl[2][2u << S1];
    const ModupJob& j = jobs[off + blockIdx.y];
    const uint32_t tid = threadIdx.x;
    // Workgroups go to the 8 XCDs in turn (linear id mod 8, and gridDim.x is
    // a multiple of 8 when remapped), each with its own L2.  A tile's rows are
    // 2^(10 - S1) words, shorter than a 128-byte L2 line at every ring size,
    // so neighbouring tiles share lines: give each XCD a run of consecutive
    // tiles of the tower instead of every eighth one.
    const uint32_t nt = gridDim.x;
    const uint32_t tile = nt % 8 ? blockIdx.x : (blockIdx.x % 8) * (nt / 8) + blockIdx.x / 8;
    switch (j.sp) {
#define GF_SP(k) \
    case k: \
        if constexpr (k <= SPMAX && (SPMAX <= 6 ? k > 0 || RS : k > 6)) modup_run<S1, k, RS, C60>(j, g, lds, twl, tid, tile); \
        break;
        GF_SP(0) GF_SP(1) GF_SP(2) GF_SP(3) GF_SP(4) GF_SP(5) GF_SP(6)
        GF_SP(7) GF_SP(8) GF_SP(9) GF_SP(10) GF_SP(11) GF_SP(12)
#undef GF_SP
    }
}

template <uint32_t SPMAX, bool RS, bool C60>
inline void run_modup(const ModupJob* d, uint32_t nj, const NttGeom& g, hipStream_t s) {
    const bool ok = with_split(g.logN1, g.logN2, [&](auto A, auto) {
        constexpr uint32_t S1 = decltype(A)::value;
        for (uint32_t off = 0; off < nj; off += MAXY) {
            const uint32_t cnt = nj - off < MAXY ? nj - off : MAXY;
            k_modup<S1, SPMAX, RS, C60><<<dim3(g.n / MODUP_TILE, cnt), MODUP_THREADS, 0, s>>>(d, off, g);
        }
    });
    if (!ok) throw std::runtime_error("gpufhe: unsupported ring dimension for the fused ModUp");
}
// jobs of 7 to 12 sources
void launch_modup_wide(const ModupJob* d, uint32_t nj, const NttGeom& g, hipStream_t s);
void launch_moddown_wide(const ModupJob* d, uint32_t nj, const NttGeom& g, hipStream_t s);

}  // namespace gf
