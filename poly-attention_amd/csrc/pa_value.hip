// pa_value.hip -- the effective value of a middle level, v * vmul rounded to the pass dtype (as the
// reference multiplies in it), as one contiguous tensor.
//
// The direct-to-LDS pass kernels move V from memory to LDS without passing it through registers, so
// they cannot multiply on the way; the register-staged kernels, which can, take 1.5 to 1.8 times as
// long.  HBM bound: two 16-byte reads and one write per 8 elements (B = 2, H = 16, N = 2048, d = 64:
// 25 MB, 7.4 us), against which a middle level at that shape saves, per launch, forward 95 -> 53 us,
// dQ 93 -> 52, dK/dV 105 -> 70 (an order-3 layer's training step at B = 8: 3083 -> 2689 us).
#include "pa_common.h"
#include "pa_launch.h"
#include "pa_mfma.h"

namespace pa {

constexpr int kValueThreads = 256;

template <typename T>
__global__ __launch_bounds__(kValueThreads) void k_value_mul(PassDev P, T* out, int hv) {
    const int cpr = P.dim / 8;
    const int64_t total = (int64_t)P.batch * hv * P.nk * cpr;
    const int64_t step = (int64_t)gridDim.x * kValueThreads;
    for (int64_t e = (int64_t)blockIdx.x * kValueThreads + threadIdx.x; e < total; e += step) {
        const int c = (int)(e % cpr);
        const int64_t row = e / cpr;
        const int j = (int)(row % P.nk);
        const int bh = (int)(row / P.nk), b = bh / hv, h = (bh % hv) * (P.heads / hv);
        const u32x4_t v = *reinterpret_cast<const u32x4_t*>(P.v.row<T>(b, h, j) + 8 * c);
        const u32x4_t m = *reinterpret_cast<const u32x4_t*>(P.vmul.row<T>(b, h, j) + 8 * c);
        *reinterpret_cast<u32x4_t*>(out + row * P.dim + 8 * c) = mul_round8<T>(v, m);
    }
}

void launch_value_mul(const PassDev& P, void* out, int hv, int dtype, hipStream_t s) {
    const int64_t chunks = (int64_t)P.batch * hv * P.nk * (P.dim / 8);
    const int64_t blocks = (chunks + kValueThreads - 1) / kValueThreads;
    const dim3 grid((uint32_t)(blocks < 8192 ? blocks : 8192));
    ProfScope ps("value_mul", s);
    if (dtype == PA_BF16)
        hipLaunchKernelGGL((k_value_mul<bf16>), grid, dim3(kValueThreads), 0, s, P, static_cast<bf16*>(out), hv);
    else
        hipLaunchKernelGGL((k_value_mul<f16>), grid, dim3(kValueThreads), 0, s, P, static_cast<f16*>(out), hv);
}

}  // namespace pa
