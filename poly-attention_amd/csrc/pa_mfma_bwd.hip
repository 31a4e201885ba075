// pa_mfma_bwd.hip -- dispatch of the 16-bit MFMA backward passes (kernels: pa_mfma_bwd.h), instantiated
// here for bf16.
#include "pa_mfma_bwd.h"

namespace pa {

bool mfma_bwd_supported(const GradDev& G, int dtype) {
    const PassDev& P = G.f;
    if (dtype == PA_F32) return mfma_bwd_f32_supported(G);
    if (dtype != PA_BF16 && dtype != PA_F16) return false;
    if (P.dim != 64 && P.dim != 128 && P.dim != 256) return false;
    const DView* loads[] = {&P.q, &P.k, &P.v, &G.dout};
    for (const DView* v : loads)
        if (!aligned_rows_host(*v, 8)) return false;
    if (P.vmul.ok() && !aligned_rows_host(P.vmul, 8)) return false;
    const DView* stores[] = {&G.dq, &G.dk, &G.dv};
    for (const DView* v : stores)
        if (!aligned_rows_host(*v, 4)) return false;
    if (P.vmul.ok() && !aligned_rows_host(G.dvmul, 4)) return false;
    return true;
}

// The preprocess folded into the direct-to-LDS dQ kernel (which then runs first): it loads
// the O rows of its queries beside dO with 16-byte loads.
bool mfma_bwd_fuses_pre(const GradDev& G) {
    const PassDev& P = G.f;
    if (!PA_BWD_DMA || P.vmul.ok() || P.q.dtype == PA_F32) return false;
    if (P.dim != 64 && P.dim != 128) return false;
    return bwd_dq_dma_ok(G) && aligned_rows_host(P.out, 8);
}

bool mfma_bwd_dma_applies(const GradDev& G) {
    return mfma_bwd_fuses_pre(G) && bwd_dma_ok(G);
}

void launch_mfma_bwd(const GradDev& G, int dtype, hipStream_t s) {
    if (dtype == PA_F32) {
        launch_mfma_bwd_f32(G, s);
        return;
    }
    if (dtype == PA_BF16) launch_bwd_dtype<bf16>(G, s);
    else launch_mfma_bwd_f16(G, s);
}

}  // namespace pa
