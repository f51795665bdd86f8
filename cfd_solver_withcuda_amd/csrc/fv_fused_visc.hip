// One-launch second-order pass with viscous terms: stages and residual mode (see fv_fused.h).
#include "fv_fused.h"

namespace cfd {

hipError_t launch_fused_visc(const FusedArgs &a, int flux, int lim, int mode, int threads, size_t sm, hipStream_t s) {
    return mode == MODE_RESID ? launch_fused_family<MODE_RESID, true, 0, false>(a, flux, lim, threads, sm, s)
                              : launch_fused_family<MODE_STAGE, true, 0, false>(a, flux, lim, threads, sm, s);
}

}  // namespace cfd
