// The fused ModUp and ModDown (modup_kernel.hpp) of up to 6 sources, and their
// launches.
#include "modup_kernel.hpp"

namespace gf {

// sp: the largest source count of the jobs, all of them at most 6 or all above
template <bool RS, bool C60>
static void launch_modup_t(const ModupJob* d, uint32_t nj, const NttGeom& g, uint32_t sp, hipStream_t s) {
    if (g.single || g.n % MODUP_TILE || (sp < 1 && !RS) || sp > (C60 ? 6u : (uint32_t)MODUP_MAXSRC))
        throw std::runtime_error("gpufhe: fused ModUp / ModDown launch shape out of range");
    if (sp <= 2) run_modup<2, RS, C60>(d, nj, g, s);
    else if (sp <= 4) run_modup<4, RS, C60>(d, nj, g, s);
    else if (sp <= 6) run_modup<6, RS, C60>(d, nj, g, s);
    else if (RS) launch_moddown_wide(d, nj, g, s);
    else launch_modup_wide(d, nj, g, s);
}
// arg: the largest source count | c60 << 8
void launch_modup(const ModupJob* d, uint32_t nj, const NttGeom& g, uint32_t arg, hipStream_t s) {
    if (arg >> 8) launch_modup_t<false, true>(d, nj, g, arg & 0xff, s);
    else launch_modup_t<false, false>(d, nj, g, arg & 0xff, s);
}
void launch_moddown(const ModupJob* d, uint32_t nj, const NttGeom& g, uint32_t sp, hipStream_t s) {
    launch_modup_t<true, false>(d, nj, g, sp, s);
}

}  // namespace gf
