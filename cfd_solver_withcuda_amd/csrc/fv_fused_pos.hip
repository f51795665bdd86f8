// One-launch second-order stages with the positivity fallback: the detecting and the recomputing
// pass (see fv_fused.h; fv_pos.hip has the two-pass form and the list of marked tiles).
#include "fv_fused.h"

namespace cfd {

hipError_t launch_fused_pos(const FusedArgs &a, int flux, int lim, int pass, int threads, size_t sm, hipStream_t s) {
    if (a.st.freeze)
        return pass == 1 ? launch_fused_family<MODE_STAGE, false, 1, true>(a, flux, lim, threads, sm, s)
                         : launch_fused_family<MODE_STAGE, false, 2, true>(a, flux, lim, threads, sm, s);
    return pass == 1 ? launch_fused_family<MODE_STAGE, false, 1, false>(a, flux, lim, threads, sm, s)
                     : launch_fused_family<MODE_STAGE, false, 2, false>(a, flux, lim, threads, sm, s);
}

}  // namespace cfd
