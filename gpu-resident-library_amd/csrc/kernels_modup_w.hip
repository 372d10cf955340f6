// The fused ModUp (and ModDown of keyswitches) of 7 to 12 sources.
#include "modup_kernel.hpp"

namespace gf {

void launch_modup_wide(const ModupJob* d, uint32_t nj, const NttGeom& g, hipStream_t s) {
    run_modup<12, false, false>(d, nj, g, s);
}

}  // namespace gf
