// The fused row pass + inner product with jobs of 5 or 6 parts.
#include "ksi_kernel.hpp"

namespace gf {

void launch_ksi_wide(const KsiJob* d, uint32_t nj, const NttGeom& g, uint32_t regions, uint32_t waves, uint32_t fin, bool big,
                     hipStream_t s) {
    run_ksi<6>(d, nj, g, regions, waves, fin, big, s);
}

}  // namespace gf
