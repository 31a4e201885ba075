// pa_mfma_f32_block.hip -- fp32 passes at head dim 128 in small grids (mfma_f32_block_applies): the forward
// and dQ with one 32-row block per workgroup; the method is pa_mfma_f32.hip's.
//
// Four waves share a block, wave w taking tiles w, w + 4, ... through an LDS region of its own, and
// nothing but the merge has a barrier.  A region holds one tensor's tile: the tensors of a product
// follow one another, each loaded while the one before it is multiplied.
// What bounds it: splitting a tile (VALU) and multiplying it take about as long, one after the
// other in a wave.  The kernels of pa_mfma_f32.hip have LDS for two tiles of two tensors there, so
// at most two waves share a block (R = C = 2), half the CUs are idle, and the row's tiles make
// twice as long a chain.  us, those and these, forward / backward (dQ here, dK/dV there in both): 8
// heads x 1024 causal 89 / 295 and 61 / 269, 8 x 512 52 / 166 and 38 / 155, 4 x 2048 162 / 541 and
// 103 / 487.  (A dK/dV of this kind stages Q twice and spills: 203 against 167 at 8 x 1024.)
#include <type_traits>

#include "pa_mfma_f32.h"

namespace pa {

constexpr int kF32Waves = 4;

// a wave's own LDS writes before its reads (and its reads before the next tile's writes)
__device__ __forceinline__ void f32_wave_sync() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    asm volatile("" ::: "memory");
}

// One 32-row tile of a tensor between global memory and a wave's region.
template <int D>
struct X3Wave {
    using L = X3<D>;
    static constexpr int RP = 64 / L::CPR, NL = kF32BN / RP;  // rows per load, loads
    float v[NL][8];
    // rows [r0, r0 + 32) of a (times m), r0 < n; zeros past n
    __device__ __forceinline__ void load(const float* a, int64_t as, const float* m, int64_t ms, int r0, int n,
                                         int lane) {
        const bool full = r0 + kF32BN <= n;
        const int f = (lane % L::CPR) * 8;
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int r = r0 + lane / L::CPR + i * RP, rr = full || r < n ? r : r0;
            const float* q = a + rr * as + f;
            float4 x = *reinterpret_cast<const float4*>(q), y = *reinterpret_cast<const float4*>(q + 4);
            if (m) {
                const float4 mx = *reinterpret_cast<const float4*>(m + rr * ms + f);
                const float4 my = *reinterpret_cast<const float4*>(m + rr * ms + f + 4);
                x = make_float4(x.x * mx.x, x.y * mx.y, x.z * mx.z, x.w * mx.w);
                y = make_float4(y.x * my.x, y.y * my.y, y.z * my.z, y.w * my.w);
            }
            const float w[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
#pragma unroll
            for (int k = 0; k < 8; ++k) v[i][k] = w[k];
        }
        if (!full) {
            keep_branch();
#pragma unroll
            for (int i = 0; i < NL; ++i)
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    if (r0 + lane / L::CPR + i * RP >= n) v[i][k] = 0.f;
        }
    }
    // the tile's planes at t; mx: the largest magnitude seen
    template <bool BIG>
    __device__ __forceinline__ void store(bf16* t, int lane, float& mx) const {
        if (!BIG)
#pragma unroll
            for (int i = 0; i < NL; ++i) mx = max_abs8(v[i], mx);
        f32_wave_sync();
#pragma unroll
        for (int i = 0; i < NL; ++i)
            L::store(t, lane / L::CPR + i * RP, lane % L::CPR, split8(v[i], BIG));
        f32_wave_sync();
    }
};

template <int D>
__global__ __launch_bounds__(64 * kF32Waves) void k_mfma_fwd_f32_block(PassDev P) {
    using L = X3<D>;
    constexpr int NW = kF32Waves;
    __shared__ __attribute__((aligned(16))) bf16 sT[NW * L::TILE];
    __shared__ float sB[NW * kF32BN];
    static_assert(sizeof(sT) >= (NW - 1) * (D / 32 * 16 + 2) * 64 * 4, "merge buffer");
    const int lane = threadIdx.x & 63, w = wave_id();
    bf16* T = sT + w * L::TILE;
    float* B = sB + w * kF32BN;
    const bool causal = P.causal != 0, sc = P.softclamp > 0.f;
    const int nqb = (P.nq + 31) / 32;
    int bh, rank;
    if (causal) block_order<true>(nqb, P.heads, P.k.hdiv, bh, rank);
    else block_order<false>(nqb, P.heads, P.k.hdiv, bh, rank);
    const int h = bh % P.heads, b = bh / P.heads;
    X3Lane<D> ln;
    ln.init(lane);
    const int q0 = (causal ? nqb - 1 - rank : rank) * 32, qi = q0 + ln.col;
    const int ntiles = ((causal ? min(P.nk, q0 + 32) : P.nk) + kF32BN - 1) / kF32BN;
    const float* kp = P.k.row<float>(b, h, 0);
    const float* vp = P.v.row<float>(b, h, 0);
    const float* mp = P.vmul.ok() ? P.vmul.row<float>(b, h, 0) : nullptr;
    f32x16_t o[D / 32];
    float m, l, big;  // big: the largest magnitude of the operands
    X3Wave<D> st;
    float rb = 0.f;
    auto load_k = [&](int t) __attribute__((always_inline)) {
        st.load(kp, P.k.sn, nullptr, 0, t * kF32BN, P.nk, lane);
        const int j = t * kF32BN + lane;
        if (lane < kF32BN) rb = j < P.nk && P.km.keep(b, j) ? key_term_l2(P, b, h, j) : -INFINITY;
    };
    auto sweep = [&](auto bigc) __attribute__((always_inline)) {
        constexpr bool BIG = decltype(bigc)::value;
        Split8 qf[D / 16];
        big = x3_load_rows<D, BIG>(P.q.row<float>(b, h, qi < P.nq ? qi : 0), nullptr, qi < P.nq, ln.hh, qf)
                  ? INFINITY : 0.f;
#pragma unroll
        for (int x = 0; x < D / 32; ++x) o[x] = zero16();
        m = -INFINITY;
        l = 0.f;
        if (w < ntiles) load_k(w);
        for (int t = w; t < ntiles; t += NW) {  // wave-uniform
            const int j0 = t * kF32BN;
            if (lane < kF32BN) B[lane] = rb;
            st.template store<BIG>(T, lane, big);
            st.load(vp, P.v.sn, mp, P.vmul.sn, j0, P.nk, lane);
            f32x16_t s = zero16();
            ln.template rows_mma<BIG>(T, qf, s);
            f32_softmax_tile<D>(P, s, B, sc, causal && j0 + 31 > q0, qi - j0 - 4 * ln.hh, ln.hh, o, m, l);
            st.template store<BIG>(T, lane, big);
            if (t + NW < ntiles) load_k(t + NW);
            ln.template cols_mma<BIG>(T, s, o);
        }
    };
    sweep(std::false_type());
    if (__builtin_expect(__any(big > kF32Split), 0)) sweep(std::true_type());  // (no barriers in a sweep)
    if (x3_merge_softmax<D, 1, NW>(o, m, l, reinterpret_cast<float*>(sT), 0, w, lane)) return;
    f32_store_out<D>(P, b, h, qi, ln.hh, o, m, l);
}

template <int D>
__global__ __launch_bounds__(64 * kF32Waves) void k_mfma_bwd_f32_dq_block(GradDev G) {
    using L = X3<D>;
    constexpr int NW = kF32Waves;
    const PassDev& P = G.f;
    __shared__ __attribute__((aligned(16))) bf16 sT[NW * L::TILE];
    __shared__ float sB[NW * kF32BN];
    static_assert(sizeof(sT) >= (NW - 1) * (D / 32 * 16 + 1) * 64 * 4, "merge buffer");
    const int lane = threadIdx.x & 63, w = wave_id();
    bf16* T = sT + w * L::TILE;
    float* B = sB + w * kF32BN;
    const bool causal = P.causal != 0, sc = P.softclamp > 0.f;
    const int nqb = (P.nq + 31) / 32;
    int bh, rank;
    if (causal) block_order<true>(nqb, P.heads, P.k.hdiv, bh, rank);
    else block_order<false>(nqb, P.heads, P.k.hdiv, bh, rank);
    const int h = bh % P.heads, b = bh / P.heads;
    X3Lane<D> ln;
    ln.init(lane);
    const int q0 = (causal ? nqb - 1 - rank : rank) * 32, qi = q0 + ln.col;
    const bool qrow = qi < P.nq;
    const int64_t r = ((int64_t)b * P.heads + h) * G.rsn + (qrow ? qi : 0);
    const float lse_l2 = qrow ? G.ws_lse[r] * kLog2e : INFINITY;
    const float dsum = qrow ? G.ws_D[r] : 0.f;
    const int ntiles = ((causal ? min(P.nk, q0 + 32) : P.nk) + kF32BN - 1) / kF32BN;
    const float* kp = P.k.row<float>(b, h, 0);
    const float* vp = P.v.row<float>(b, h, 0);
    const float* mp = P.vmul.ok() ? P.vmul.row<float>(b, h, 0) : nullptr;
    f32x16_t dq[D / 32];
    float big;  // the largest magnitude of the operands
    X3Wave<D> st;
    auto load_v = [&](int t) __attribute__((always_inline)) {
        st.load(vp, P.v.sn, mp, P.vmul.sn, t * kF32BN, P.nk, lane);
    };
    auto sweep = [&](auto bigc) __attribute__((always_inline)) {
        constexpr bool BIG = decltype(bigc)::value;
        Split8 qf[D / 16], of[D / 16];
        const bool bq = x3_load_rows<D, BIG>(P.q.row<float>(b, h, qrow ? qi : 0), nullptr, qrow, ln.hh, qf);
        const bool bo = x3_load_rows<D, BIG>(G.dout.row<float>(b, h, qrow ? qi : 0), nullptr, qrow, ln.hh, of);
        big = bq || bo ? INFINITY : 0.f;
#pragma unroll
        for (int x = 0; x < D / 32; ++x) dq[x] = zero16();
        if (w < ntiles) load_v(w);
        for (int t = w; t < ntiles; t += NW) {  // wave-uniform
            const int j0 = t * kF32BN;
            st.template store<BIG>(T, lane, big);
            st.load(kp, P.k.sn, nullptr, 0, j0, P.nk, lane);
            const float rb = key_term_l2(P, b, h, j0 + ln.col);
            f32x16_t s = zero16(), dp = zero16();
            ln.template rows_mma<BIG>(T, of, dp);
            if (lane < kF32BN) B[lane] = rb;
            st.template store<BIG>(T, lane, big);
            if (t + NW < ntiles) load_v(t + NW);
            ln.template rows_mma<BIG>(T, qf, s);
            f32_ds_query<D>(P, s, dp, B, sc, causal ? qi - j0 - 4 * ln.hh : 1 << 30, ln.hh, lse_l2, dsum);
            if (!BIG) big = max_abs16(s, big);
            ln.template cols_mma<BIG>(T, s, dq);
        }
    };
    sweep(std::false_type());
    if (__builtin_expect(__any(big > kF32Split), 0)) sweep(std::true_type());
    {
        f32x16_t* acc[D / 32];
#pragma unroll
        for (int x = 0; x < D / 32; ++x) acc[x] = &dq[x];
        float none = 0.f;
        if (x3_merge<D / 32, 1, NW>(acc, &none, reinterpret_cast<float*>(sT), 0, w, lane)) return;
    }
    if (qrow) f32_store_dq<D>(G, b, h, qi, ln.hh, dq);
}

// Head dim 128, at most one 32-row block per CU (causal grids, whose blocks differ in length: three for
// two) and four stages of two tiles or more.  With fewer tiles their fixed part costs as much (us
// forward / backward at 8 heads x 64: 19.6 / 60.3, these 20.6 / 61.5); in larger grids a CU's second
// block waits for its first (3 x 8 heads x 512, 384 blocks: causal 54 / 179, these 48 / 180, not causal
// 55 / 177, these 69 / 213; 1024 blocks, causal: 106 / 373, these 144 / 460).
bool mfma_f32_block_applies(const PassDev& P, int64_t blocks) {
    return P.dim == 128 && blocks <= (P.causal ? 384 : 256) && P.nk > 7 * kF32BN;
}

void launch_mfma_fwd_f32_block(const PassDev& P, int64_t blocks, hipStream_t s) {
    ProfScope ps("mfma_fwd_f32_split", s);
    hipLaunchKernelGGL((k_mfma_fwd_f32_block<128>), dim3((uint32_t)blocks), dim3(64 * kF32Waves), 0, s, P);
}

void launch_mfma_bwd_f32_dq_block(const GradDev& G, int64_t blocks, hipStream_t s) {
    ProfScope ps("mfma_bwd_f32_dq_split", s);
    hipLaunchKernelGGL((k_mfma_bwd_f32_dq_block<128>), dim3((uint32_t)blocks), dim3(64 * kF32Waves), 0, s, G);
}

}  // namespace pa
