// One-launch second-order stages with limiter freezing, inviscid and viscous (see fv_fused.h).
#include "fv_fused.h"

namespace cfd {

hipError_t launch_fused_freeze(const FusedArgs &a, int flux, int lim, bool visc, int threads, size_t sm, hipStream_t s) {
    return visc ? launch_fused_family<MODE_STAGE, true, 0, true>(a, flux, lim, threads, sm, s)
                : launch_fused_family<MODE_STAGE, false, 0, true>(a, flux, lim, threads, sm, s);
}

}  // namespace cfd
