// pa_mfma_bwd_f16.hip -- the 16-bit MFMA backward kernels (pa_mfma_bwd.h) for f16.
#include "pa_mfma_bwd.h"

namespace pa {

void launch_mfma_bwd_f16(const GradDev& G, hipStream_t s) { launch_bwd_dtype<f16>(G, s); }

}  // namespace pa
