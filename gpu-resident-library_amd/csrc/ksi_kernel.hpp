// The fused row pass of the keyswitch digits' forward transform and the key
// inner product (ksi.hpp), with its launch.
#pragma once
#include "ksi.hpp"
#include "ntt_kernels.hpp"

namespace gf {

// ------------------------------------------- fused digit row pass + inner --
// One wave's LDS region is private to it during the row passes.
struct WaveSync {
    __device__ void operator()() const { DevSync{}.wave(); }
    __device__ void wave() const { DevSync{}.wave(); }
};

// At most 96 VGPRs (5 waves per SIMD, 20 per CU): every phase waits on memory
// (row passes for twiddles, inner products for digits and keys), so the waves
// in flight set the time.  Four parts with their last step take 5 waves of
// 107 VGPRs uncapped: 64 EvalMult+Rescale at n = 2^16, L = 24 ran 8300 us with 4
// waves per SIMD, 7570 with 5, 8280 with 6 (spills).  The last step's kernels
// (NPMAX = 4) spill scalar registers into vector lanes, 33 to 41 in KSI_FIN, none
// to 6 with the tensor products, and there 1 to 5 VGPRs to scratch; the stored
// form spills nothing.
// FIN: KSI_PLAIN, KSI_FIN, KSI_FIN_TENSOR(_IN); NPMAX: the largest part count with
// column sums (4, or 6 in kernels_ksi_w.hip).
template <uint32_t S2, uint32_t RM, int FIN, int NPMAX, uint32_t LOGT = KSI_LOG_TILE>
__global__ __launch_bounds__(KSI_THREADS) __attribute__((amdgpu_waves_per_eu(5, 8))) void k_ksi(const KsiJob* __restrict__ jobs, uint32_t off, uint32_t N1) {
    extern __shared__ __align__(16) uint64_t lds[];
    const KsiJob& j = jobs[off + blockIdx.y];
    const uint32_t tid = threadIdx.x, nthr = blockDim.x;
    auto go = [&](auto L) {
        ksi_body<S2, RM, decltype(L)::value, WaveSync, DevSync, FIN, NPMAX, LOGT>(
            j, N1, blockIdx.x, lds, tid >> 6, nthr >> 6, tid & 63, 64, tid, nthr, WaveSync{}, DevSync{});
    };
    if (j.red) go(std::true_type{});
    else go(std::false_type{});
}

template <int NPMAX>
inline void run_ksi(const KsiJob* d, uint32_t nj, const NttGeom& g, uint32_t regions, uint32_t waves, uint32_t fin,
                    bool big, hipStream_t s) {
    if (big) {
        const size_t shm = (size_t)regions * ksi_part_words(KSI_LOG_TILE_BIG) * 8;
        const bool ok = with_split(g.logN1, g.logN2, [&](auto, auto B) {
            for (uint32_t off = 0; off < nj; off += MAXY)
                k_ksi<decltype(B)::value, 4, KSI_PLAIN, NPMAX, KSI_LOG_TILE_BIG>
                    <<<dim3(g.n >> KSI_LOG_TILE_BIG, nj - off < MAXY ? nj - off : MAXY), 64 * waves, shm, s>>>(d, off, 1u << g.logN1);
        });
        if (!ok) throw std::runtime_error("gpufhe: unsupported ring dimension for the NTT");
        return;
    }
    // The input towers through LDS: 64 EvalMult+Rescale at n = 2^16, L = 24 6970 ->
    // 6780 us, one 196 -> 192; as a run-time branch of one kernel 6906 (spills).
    // The inputs' 16 KiB take no workgroup per CU from launches of 5 regions (4 of
    // 5 waves, 37.3 of 160 KiB each).  Launches of 4 would lose one of 5 and run
    // no faster (chains of three parts 2797 -> 2814 us, two parts 157.3 -> 159.7).
    const bool in = fin == KSI_FIN_TENSOR && (NPMAX > 4 || regions >= 5);
    const size_t shm = ((size_t)regions * KSI_PART_WORDS + (in ? KSI_IN_WORDS : 0)) * 8;
    bool ok = with_row_radix(g.rmax, [&](auto Rc) {
        constexpr uint32_t RM = decltype(Rc)::value;
        const bool geom_ok = with_split(g.logN1, g.logN2, [&](auto, auto B) {
            constexpr uint32_t S2 = decltype(B)::value;
            for (uint32_t off = 0; off < nj; off += MAXY) {
                const uint32_t cnt = nj - off < MAXY ? nj - off : MAXY;
                const dim3 grid(g.n / KSI_TILE, cnt);
                const uint32_t N1 = 1u << g.logN1;
                if (in) k_ksi<S2, RM, KSI_FIN_TENSOR_IN, NPMAX><<<grid, 64 * waves, shm, s>>>(d, off, N1);
                else if (fin == KSI_FIN_TENSOR)
                    k_ksi<S2, RM, NPMAX == 4 ? KSI_FIN_TENSOR : KSI_FIN_TENSOR_IN, NPMAX><<<grid, 64 * waves, shm, s>>>(d, off, N1);
                else if (fin) k_ksi<S2, RM, KSI_FIN, NPMAX><<<grid, 64 * waves, shm, s>>>(d, off, N1);
                else k_ksi<S2, RM, KSI_PLAIN, NPMAX><<<grid, 64 * waves, shm, s>>>(d, off, N1);
            }
        });
        if (!geom_ok) throw std::runtime_error("gpufhe: unsupported ring dimension for the NTT");
    });
    if (!ok) throw std::runtime_error("gpufhe: unsupported NTT radix");
}
// launches with jobs of 5 or 6 parts
void launch_ksi_wide(const KsiJob* d, uint32_t nj, const NttGeom& g, uint32_t regions, uint32_t waves, uint32_t fin, bool big,
                     hipStream_t s);

}  // namespace gf
