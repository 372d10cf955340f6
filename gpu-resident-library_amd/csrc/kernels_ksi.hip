// The fused row pass of the keyswitch digits and the key inner product
// (ksi_kernel.hpp), with its launch.
#include "ksi_kernel.hpp"

namespace gf {

void launch_ksi(const KsiJob* d, uint32_t nj, const NttGeom& g, uint32_t regions, uint32_t waves, uint32_t fin, bool wide,
                bool big, hipStream_t s) {
    if (g.single || g.n % KSI_TILE) throw std::runtime_error("gpufhe: fused inner product needs a two-phase ring");
    if (regions > KSI_MAXP || waves < 1 || waves > KSI_WAVES)
        throw std::runtime_error("gpufhe: fused inner product launch shape out of range");
    if (big && (fin || g.rmax != 4)) throw std::runtime_error("gpufhe: fused inner product launch shape out of range");
    if (wide) launch_ksi_wide(d, nj, g, regions, waves, fin, big, s);
    else run_ksi<4>(d, nj, g, regions, waves, fin, big, s);
}

}  // namespace gf
