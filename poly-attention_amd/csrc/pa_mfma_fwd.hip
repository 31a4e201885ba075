// pa_mfma_fwd.hip -- dispatch of the 16-bit MFMA forward passes (kernels: pa_mfma_fwd.h), instantiated
// here for bf16.
#include "pa_mfma_fwd.h"

namespace pa {

bool mfma_fwd_supported(const PassDev& P, int dtype) {
    if (dtype == PA_F32) return mfma_fwd_f32_supported(P);
    if (dtype != PA_BF16 && dtype != PA_F16) return false;
    if (P.dim != 64 && P.dim != 128 && P.dim != 256) return false;
    if (!(P.scale > 0.f)) return false;  // the raw-score running max assumes a positive scale
    if (!aligned_rows_host(P.q, 8) || !aligned_rows_host(P.k, 8) || !aligned_rows_host(P.v, 8)) return false;
    if (P.vmul.ok() && !aligned_rows_host(P.vmul, 8)) return false;
    if (!aligned_rows_host(P.out, 4)) return false;
    // the epilogue's root / gate / y rows travel in 8-byte words
    for (const DView* e : {&P.er, &P.eg, &P.ey})
        if (e->ok() && !aligned_rows_host(*e, 4)) return false;
    return true;
}

bool mfma_fwd_short_applies(const PassDev& P, int dtype) {
    return PA_FWD_SHORT && (dtype == PA_BF16 || dtype == PA_F16) && P.dim == 64 && !P.causal &&
           !P.vmul.ok() && P.nq <= 64 && P.nk <= 64 && !P.km.p;
}

bool mfma_fwd_dma_applies(const PassDev& P) {
    return (P.dim == 64 || P.dim == 128) && !P.vmul.ok() && dma_ok(P, 64);
}

void launch_mfma_fwd(const PassDev& P, int dtype, hipStream_t s) {
    if (dtype == PA_F32) {
        launch_mfma_fwd_f32(P, s);
        return;
    }
    if (dtype == PA_BF16) launch_fwd_t<bf16>(P, s);
    else launch_mfma_fwd_f16(P, s);
}

bool mfma_order2_short_applies(const PassDev& P1, const PassDev& P2, int dtype) {
    if (!(dtype == PA_BF16 || dtype == PA_F16)) return false;
    if (!mfma_fwd_supported(P1, dtype) || !mfma_fwd_supported(P2, dtype)) return false;
    if (!mfma_fwd_short_applies(P1, dtype) || !mfma_fwd_short_applies(P2, dtype)) return false;
    if (P1.batch != P2.batch || P1.heads != P2.heads || P2.nk != P1.nq) return false;
    if ((P1.softclamp > 0.f) != (P2.softclamp > 0.f)) return false;
    // pass 1 has no key term and no epilogue; no query masks
    if (P1.bias.ok() || P1.ey.ok() || P1.qm.p || P2.qm.p) return false;
    // q2 is normalised once: pass 2's key norm must be pass 1's query norm
    const bool nq1 = (P1.nflags & PA_NORM_Q) != 0, nk2 = (P2.nflags & PA_NORM_K) != 0;
    if (nq1 != nk2) return false;
    if (nq1 && (P1.qnw != P2.knw || P1.qeps != P2.keps)) return false;
    return true;
}

void launch_order2_short(const PassDev& P1, const PassDev& P2, int dtype, hipStream_t s) {
    if (dtype == PA_BF16) launch_o2<bf16>(P1, P2, s);
    else launch_order2_short_f16(P1, P2, s);
}

}  // namespace pa
