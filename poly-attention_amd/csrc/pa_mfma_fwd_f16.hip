// pa_mfma_fwd_f16.hip -- the 16-bit MFMA forward kernels (pa_mfma_fwd.h) for f16.
#include "pa_mfma_fwd.h"

namespace pa {

void launch_mfma_fwd_f16(const PassDev& P, hipStream_t s) { launch_fwd_t<f16>(P, s); }

void launch_order2_short_f16(const PassDev& P1, const PassDev& P2, hipStream_t s) {
    launch_o2<f16>(P1, P2, s);
}

}  // namespace pa
