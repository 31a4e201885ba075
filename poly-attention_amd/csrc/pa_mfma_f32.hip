// pa_mfma_f32.hip -- fp32 attention passes on the bf16 matrix cores (gfx950), head dim 64 or 128: the
// forward (every pass feature), and the backward of unmasked passes.
//
// Every fp32 operand is split into three bf16 numbers, x = h + m + l (each the rounding of what the
// ones before it leave: 8 + 8 + 8 significant bits, exact from 2^-110 up, where l reaches bf16's
// smallest number 2^-133; smaller x lose low bits), and a product x y is the six of the nine
// partial products above 2^-26 of it: h h, h m, m h, m m, h l, l h, summed small ones first into the
// fp32 accumulators of v_mfma_f32_32x32x16_bf16.  That is 6
// instructions of 32 cycles per 32 x 32 x 16 product against 8 of 64 cycles on v_mfma_f32_32x32x2_f32
// (192 and 512 cycles), reads each LDS operand as 16-byte fragments instead of one scalar per
// instruction, and rounds the accumulator 6 times per 16 terms instead of 16.  Against 64 bits it
// is closer than the fp32 instruction: largest relative error of out and the gradients 5.8e-7
// against 1.1e-6 (B = 2, H = 8, N = 1024, d = 64, causal, order-2 forward and backward).
//
// A workgroup of R * C waves owns R blocks of 32 rows (queries in the forward and dQ, keys in
// dK/dV); wave (r, c) takes row block r and every C-th tile of 32 rows of the other side.  The C
// tiles of a stage travel through registers (the next stage's loads are in flight while this one
// is computed), are split once and stored as three bf16 planes in LDS, row-major with 16-byte
// chunks XOR-swizzled, which serve both the row fragments (ds_read_b128) and the transposed ones
// (ds_read_b64_tr_b16).  The C waves of a row block merge their results at the end, in order.
//   S^T = K Q^T and O^T += V^T P^T as in the 16-bit kernels (pa_mfma.h): lane l holds query
//   l % 32 and the probabilities enter the second product from the score registers, split there.
// What bounds it: at R C = 8 waves (two per SIMD) the matrix cores and the VALU (splitting the
// staged tiles and P, the softmax) about equally.  C > 1 is for small grids: 512 blocks of 32 rows
// (B = 2, H = 8, N = 1024) are 512 waves on 1024 SIMDs without it, the heaviest of a causal grid
// 32 tiles long.
// Measured per level at B = 2, H = 8, N = 1024, d = 64, causal, against one-wave workgroups on the fp32
// instruction: forward 134 -> 41 us, dQ 175 -> 55, dK/dV 211 -> 60; B = 4, H = 16, N = 2048: forward
// 210 us, 164 TFLOP/s (the fp32 instruction's peak is 157).
//
// Infinities: x = inf splits into (inf, 0, 0), whose small partial products would be inf * 0 = NaN. A
// workgroup that has met one (or a number that rounds to one in bf16) sweeps its tiles again, with
// every infinite h taken as 0 in the small products: h h alone then gives what the fp32 product
// gives; where waves have no barrier in a sweep (pa_mfma_f32_block.hip) each decides for itself. (A branch
// in each tile instead cost the backward kernels up to 200 spilled registers.)
// Masks, key bias classes, value multiplier, softclamp, causal limits and
// the module epilogue follow the pass semantics of polyattn.h; rows left fully masked get lse = NaN
// for k_fwd_fixup, as in the 16-bit kernels.
#include "pa_mfma_f32.h"

namespace pa {

// A stage of C tiles of two [n, D] fp32 tensors between global memory and LDS.
template <int D, int NT, int C>
struct X3Stage {
    using L = X3<D>;
    static constexpr int CH = C * kF32BN * L::CPR;  // 8-float chunks per tensor
    static constexpr int NL = 2 * CH / NT;          // chunks per thread
    static_assert(CH % NT == 0 || NT % CH == 0, "a thread's chunks are of one tensor each");
    static_assert(NL >= 1 && 2 * CH % NT == 0, "whole chunks per thread");
    float v[NL][8];
    // rows [r0, r0 + 32 C) of a and of c (times m), zeros past n
    __device__ __forceinline__ void load(const float* a, int64_t as, const float* c, int64_t cs,
                                         const float* m, int64_t ms, int r0, int n) {
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int p = threadIdx.x + i * NT, e = p % CH, r = r0 + e / L::CPR, f = (e % L::CPR) * 8;
            const bool second = p >= CH, ok = r < n;
            const int64_t rr = ok ? r : 0;
            const float* q = second ? c + rr * cs + f : a + rr * as + f;
            float4 x = *reinterpret_cast<const float4*>(q), y = *reinterpret_cast<const float4*>(q + 4);
            if (m && second) {
                const float4 mx = *reinterpret_cast<const float4*>(m + rr * ms + f);
                const float4 my = *reinterpret_cast<const float4*>(m + rr * ms + f + 4);
                x = make_float4(x.x * mx.x, x.y * mx.y, x.z * mx.z, x.w * mx.w);
                y = make_float4(y.x * my.x, y.y * my.y, y.z * my.z, y.w * my.w);
            }
            const float w[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
#pragma unroll
            for (int k = 0; k < 8; ++k) v[i][k] = ok ? w[k] : 0.f;
        }
    }
    // tiles of the first tensor at sa, of the second at sc; mx: the largest magnitude seen
    template <bool BIG>
    __device__ __forceinline__ void store(bf16* sa, bf16* sc, float& mx) const {
        if (!BIG)
#pragma unroll
            for (int i = 0; i < NL; ++i) mx = max_abs8(v[i], mx);
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int p = threadIdx.x + i * NT, e = p % CH, r = e / L::CPR;
            bf16* t = (p >= CH ? sc : sa) + (r / kF32BN) * L::TILE;
            L::store(t, r % kF32BN, e % L::CPR, split8(v[i], BIG));
        }
    }
};

// ---------------------------------------------------------------------------------------
// forward

template <int D, int R, int C>
__global__ __launch_bounds__(64 * R * C, R * C / 4) void k_mfma_fwd_f32(PassDev P) {
    using L = X3<D>;
    constexpr int NT = 64 * R * C;
    constexpr int NO = D / 32 * 16;  // accumulator registers
    __shared__ __attribute__((aligned(16))) bf16 sT[2 * C * L::TILE];
    __shared__ float sB[C * kF32BN];  // key term in log2 units: bias * log2e, -inf when masked
    __shared__ int sF;                // a value of the stage does not split
    static_assert(sizeof(sT) >= (size_t)R * (C - 1) * (NO + 2) * 64 * 4, "merge buffer");
    bf16* sK = sT;
    bf16* sV = sT + C * L::TILE;

    const int tid = threadIdx.x, lane = tid & 63, w = wave_id(), wr = w / C, wc = w % C;
    const bool causal = P.causal != 0;
    const int nqb = (P.nq + 32 * R - 1) / (32 * R);
    int bh, rank;
    if (causal) block_order<true>(nqb, P.heads, P.k.hdiv, bh, rank);
    else block_order<false>(nqb, P.heads, P.k.hdiv, bh, rank);
    const int qb = causal ? nqb - 1 - rank : rank;
    const int h = bh % P.heads, b = bh / P.heads;
    X3Lane<D> ln;
    ln.init(lane);
    const int q0 = (qb * R + wr) * 32, qi = q0 + ln.col;

    f32x16_t o[D / 32];
    float m, l, big;  // big: the largest magnitude of the operands

    const bool sc = P.softclamp > 0.f;
    const int kend = causal ? min(P.nk, (qb + 1) * 32 * R) : P.nk;
    const int wave_kend = causal ? min(kend, q0 + 32) : kend;
    const float* kp = P.k.row<float>(b, h, 0);
    const float* vp = P.v.row<float>(b, h, 0);
    const float* mp = P.vmul.ok() ? P.vmul.row<float>(b, h, 0) : nullptr;

    X3Stage<D, NT, C> st;
    float rb = 0.f;
    auto load = [&](int j0) __attribute__((always_inline)) {
        st.load(kp, P.k.sn, vp, P.v.sn, mp, P.vmul.sn, j0, P.nk);
        if (tid < C * kF32BN) {
            const int j = j0 + tid;
            rb = j < P.nk && P.km.keep(b, j) ? key_term_l2(P, b, h, j) : -INFINITY;
        }
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
        if (kend > 0) load(0);
        for (int s0 = 0; s0 < kend; s0 += C * kF32BN) {
            __syncthreads();
            st.template store<BIG>(sK, sV, big);
            if (tid < C * kF32BN) sB[tid] = rb;
            __syncthreads();
            if (s0 + C * kF32BN < kend) load(s0 + C * kF32BN);
            const int j0 = s0 + wc * kF32BN;
            if (j0 < wave_kend) {  // wave-uniform: the causal limit of this wave's queries
                const bf16* K = sK + wc * L::TILE;
                const bf16* V = sV + wc * L::TILE;
                const float* B = sB + wc * kF32BN;
                f32x16_t s = zero16();
                ln.template rows_mma<BIG>(K, qf, s);
                f32_softmax_tile<D>(P, s, B, sc, causal && j0 + 31 > q0, qi - j0 - 4 * ln.hh, ln.hh, o, m, l);
                ln.template cols_mma<BIG>(V, s, o);
            }
        }
    };
    sweep(std::false_type());
    if (__builtin_expect(x3_met_big(big, &sF), 0)) sweep(std::true_type());
    if (x3_merge_softmax<D, R, C>(o, m, l, reinterpret_cast<float*>(sT), wr, wc, lane)) return;
    f32_store_out<D>(P, b, h, qi, ln.hh, o, m, l);
}

// ---------------------------------------------------------------------------------------
// backward (unmasked passes; after the row preprocess: ws_lse, ws_D)

// dQ, query-major: S^T = K Q^T and dP^T = V dO^T (lane = query), dS, then dQ^T += K^T dS^T with dS
// entering as B.
template <int D, int R, int C>
__global__ __launch_bounds__(64 * R * C, R * C / 4) void k_mfma_bwd_f32_dq(GradDev G) {
    using L = X3<D>;
    constexpr int NT = 64 * R * C;
    const PassDev& P = G.f;
    __shared__ __attribute__((aligned(16))) bf16 sT[2 * C * L::TILE];
    __shared__ float sB[C * kF32BN];
    __shared__ int sF;
    static_assert(sizeof(sT) >= (size_t)R * (C - 1) * (D / 32 * 16 + 1) * 64 * 4, "merge buffer");
    bf16* sK = sT;
    bf16* sV = sT + C * L::TILE;
    const int tid = threadIdx.x, lane = tid & 63, w = wave_id(), wr = w / C, wc = w % C;
    const bool causal = P.causal != 0;
    const int nqb = (P.nq + 32 * R - 1) / (32 * R);
    int bh, rank;
    if (causal) block_order<true>(nqb, P.heads, P.k.hdiv, bh, rank);
    else block_order<false>(nqb, P.heads, P.k.hdiv, bh, rank);
    const int qb = causal ? nqb - 1 - rank : rank;
    const int h = bh % P.heads, b = bh / P.heads;
    X3Lane<D> ln;
    ln.init(lane);
    const int q0 = (qb * R + wr) * 32, qi = q0 + ln.col;
    const bool qrow = qi < P.nq;
    const int64_t r = ((int64_t)b * P.heads + h) * G.rsn + (qrow ? qi : 0);
    const float lse_l2 = qrow ? G.ws_lse[r] * kLog2e : INFINITY;
    const float dsum = qrow ? G.ws_D[r] : 0.f;
    f32x16_t dq[D / 32];
    float big;  // the largest magnitude of the operands
    const bool sc = P.softclamp > 0.f;
    const int kend = causal ? min(P.nk, (qb + 1) * 32 * R) : P.nk;
    const int wave_kend = causal ? min(kend, q0 + 32) : kend;
    const float* kp = P.k.row<float>(b, h, 0);
    const float* vp = P.v.row<float>(b, h, 0);
    const float* mp = P.vmul.ok() ? P.vmul.row<float>(b, h, 0) : nullptr;
    X3Stage<D, NT, C> st;
    float rb = 0.f;
    auto load = [&](int j0) __attribute__((always_inline)) {
        st.load(kp, P.k.sn, vp, P.v.sn, mp, P.vmul.sn, j0, P.nk);
        if (tid < C * kF32BN) rb = key_term_l2(P, b, h, j0 + tid);
    };
    auto sweep = [&](auto bigc) __attribute__((always_inline)) {
        constexpr bool BIG = decltype(bigc)::value;
        Split8 qf[D / 16], of[D / 16];
        const bool bq = x3_load_rows<D, BIG>(P.q.row<float>(b, h, qrow ? qi : 0), nullptr, qrow, ln.hh, qf);
        const bool bo = x3_load_rows<D, BIG>(G.dout.row<float>(b, h, qrow ? qi : 0), nullptr, qrow, ln.hh, of);
        big = bq || bo ? INFINITY : 0.f;
#pragma unroll
        for (int x = 0; x < D / 32; ++x) dq[x] = zero16();
        if (kend > 0) load(0);
        for (int s0 = 0; s0 < kend; s0 += C * kF32BN) {
            __syncthreads();
            st.template store<BIG>(sK, sV, big);
            if (tid < C * kF32BN) sB[tid] = rb;
            __syncthreads();
            if (s0 + C * kF32BN < kend) load(s0 + C * kF32BN);
            const int j0 = s0 + wc * kF32BN;
            if (j0 >= wave_kend) continue;  // wave-uniform; the barriers are at the loop's start
            const bf16* K = sK + wc * L::TILE;
            const bf16* V = sV + wc * L::TILE;
            const float* B = sB + wc * kF32BN;
            f32x16_t s = zero16(), dp = zero16();
            ln.template rows_mma<BIG>(K, qf, s);
            ln.template rows_mma<BIG>(V, of, dp);
            f32_ds_query<D>(P, s, dp, B, sc, causal ? qi - j0 - 4 * ln.hh : 1 << 30, ln.hh, lse_l2, dsum);
            if (!BIG) big = max_abs16(s, big);
            ln.template cols_mma<BIG>(K, s, dq);
        }
    };
    sweep(std::false_type());
    if (__builtin_expect(x3_met_big(big, &sF), 0)) sweep(std::true_type());
    {
        f32x16_t* acc[D / 32];
#pragma unroll
        for (int x = 0; x < D / 32; ++x) acc[x] = &dq[x];
        float none = 0.f;
        if (x3_merge<D / 32, R, C>(acc, &none, reinterpret_cast<float*>(sT), wr, wc, lane)) return;
    }
    if (qrow) f32_store_dq<D>(G, b, h, qi, ln.hh, dq);
}

// dK / dV / dbias, key-major: the wave's 32 keys (K and the effective value as B operands) against
// the query tiles of every query head of the group: S = Q K^T and dP = dO V^T (lane = key),
// dV^T += dO^T P and dK^T += Q^T dS with P / dS entering as B.
template <int D, int R, int C>
__global__ __launch_bounds__(64 * R * C, R * C / 4) void k_mfma_bwd_f32_dkv(GradDev G) {
    using L = X3<D>;
    constexpr int NT = 64 * R * C;
    const PassDev& P = G.f;
    constexpr int MERGE = R * (C - 1) * (2 * (D / 32) * 16 + 1) * 64 * 2;  // elements of the merge buffer
    __shared__ __attribute__((aligned(16))) bf16 sT[2 * C * L::TILE > MERGE ? 2 * C * L::TILE : MERGE];
    __shared__ float sL[C * kF32BN], sD[C * kF32BN];
    __shared__ int sF;
    bf16* sQ = sT;
    bf16* sO = sT + C * L::TILE;
    const int tid = threadIdx.x, lane = tid & 63, w = wave_id(), wr = w / C, wc = w % C;
    const bool causal = P.causal != 0;
    const int nkb = (P.nk + 32 * R - 1) / (32 * R);
    int unit, kblk;  // causal: the first key blocks carry the most work
    if (causal) block_order<true>(nkb, G.hk, 1, unit, kblk);
    else block_order<false>(nkb, G.hk, 1, unit, kblk);
    const int kh = unit % G.hk, b = unit / G.hk;
    const int rep = P.heads / G.hk, h0 = kh * rep;
    X3Lane<D> ln;
    ln.init(lane);
    const int k0 = (kblk * R + wr) * 32, kj = k0 + ln.col;
    const bool krow = kj < P.nk;
    const float bk = key_term_l2(P, b, h0, kj);  // -inf past nk
    f32x16_t dk[D / 32], dv[D / 32];
    float dbias, big;  // big: the largest magnitude of the operands
    const bool sc = P.softclamp > 0.f;
    // stages of C query tiles, from the first that reaches a key of the workgroup, head by head
    const int i_start = causal ? kblk * R * 32 : 0;
    const int nst = P.nq > i_start ? (P.nq - i_start + C * kF32BN - 1) / (C * kF32BN) : 0;
    X3Stage<D, NT, C> st;
    float rl = 0.f, rd = 0.f;
    auto load = [&](int hr, int i0) __attribute__((always_inline)) {
        const int h = h0 + hr;
        const int64_t row0 = ((int64_t)b * P.heads + h) * G.rsn;
        st.load(P.q.row<float>(b, h, 0), P.q.sn, G.dout.row<float>(b, h, 0), G.dout.sn, nullptr, 0, i0,
                P.nq);
        if (tid < C * kF32BN) {
            const int i = i0 + tid;
            rl = i < P.nq ? G.ws_lse[row0 + i] * kLog2e : INFINITY;
            rd = i < P.nq ? G.ws_D[row0 + i] : 0.f;
        }
    };
    const int total = nst * rep;
    auto sweep = [&](auto bigc) __attribute__((always_inline)) {
        constexpr bool BIG = decltype(bigc)::value;
        Split8 kf[D / 16], vf[D / 16];
        const bool bk_ = x3_load_rows<D, BIG>(P.k.row<float>(b, h0, krow ? kj : 0), nullptr, krow, ln.hh, kf);
        const bool bv_ = x3_load_rows<D, BIG>(P.v.row<float>(b, h0, krow ? kj : 0),
                                              P.vmul.ok() ? P.vmul.row<float>(b, h0, krow ? kj : 0) : nullptr,
                                              krow, ln.hh, vf);
        big = bk_ || bv_ ? INFINITY : 0.f;
#pragma unroll
        for (int x = 0; x < D / 32; ++x) {
            dk[x] = zero16();
            dv[x] = zero16();
        }
        dbias = 0.f;
        int hr = 0, s0 = i_start;  // the stage being computed
        for (int it = 0; it < total; ++it) {
            // (loaded here and not a stage ahead: the registers hold K, V, dK and dV)
            load(hr, s0);
            __syncthreads();
            st.template store<BIG>(sQ, sO, big);
            if (tid < C * kF32BN) {
                sL[tid] = rl;
                sD[tid] = rd;
            }
            __syncthreads();
            const int i0 = s0 + wc * kF32BN;
            s0 += C * kF32BN;
            if (s0 >= P.nq) {
                s0 = i_start;
                ++hr;
            }
            // wave-uniform: no query of the tile reaches a key of the wave, or past the last query
            if (i0 >= P.nq || (causal && i0 + kF32BN - 1 < k0)) continue;
            const bf16* Q = sQ + wc * L::TILE;
            const bf16* O = sO + wc * L::TILE;
            f32x16_t s = zero16(), dp = zero16();
            ln.template rows_mma<BIG>(Q, kf, s);
            ln.template rows_mma<BIG>(O, vf, dp);
            const int lim = causal ? kj - i0 - 4 * ln.hh : -(1 << 30);
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const float4 lv = *reinterpret_cast<const float4*>(sL + wc * kF32BN + 8 * g + 4 * ln.hh);
                const float4 dv4 = *reinterpret_cast<const float4*>(sD + wc * kF32BN + 8 * g + 4 * ln.hh);
                const float L4[4] = {lv.x, lv.y, lv.z, lv.w}, D4[4] = {dv4.x, dv4.y, dv4.z, dv4.w};
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int i = 4 * g + k;
                    float y = s[i] * P.scale;
                    if (sc) y = softclamp_f(y, P.softclamp);
                    float t = y * kLog2e + bk;
                    if (8 * g + k < lim) t = -INFINITY;
                    const float p = fast_exp2(t - L4[k]);
                    float ds = p * (dp[i] - D4[k]);
                    dbias += ds;
                    if (sc) ds *= softclamp_grad(y, P.softclamp);
                    s[i] = p;
                    dp[i] = ds * P.scale;
                }
            }
            if (!BIG) big = max_abs16(dp, max_abs16(s, big));
            ln.template cols_mma<BIG>(O, s, dv);
            ln.template cols_mma<BIG>(Q, dp, dk);
        }
    };
    sweep(std::false_type());
    if (__builtin_expect(x3_met_big(big, &sF), 0)) sweep(std::true_type());
    {
        f32x16_t* acc[2 * (D / 32)];
#pragma unroll
        for (int x = 0; x < D / 32; ++x) {
            acc[x] = &dk[x];
            acc[D / 32 + x] = &dv[x];
        }
        if (x3_merge<2 * (D / 32), R, C>(acc, &dbias, reinterpret_cast<float*>(sT), wr, wc, lane)) return;
    }
    dbias = xhalf_sum(dbias);
    if (!krow) return;
    const float* mr = P.vmul.ok() ? P.vmul.row<float>(b, h0, kj) : nullptr;
    const float* vr = P.v.row<float>(b, h0, kj);
    float* dkr = G.dk.wrow<float>(b, h0, kj);
    float* dvr = G.dv.wrow<float>(b, h0, kj);
    float* dmr = mr ? G.dvmul.wrow<float>(b, h0, kj) : nullptr;
#pragma unroll
    for (int x = 0; x < D / 32; ++x)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int d = 32 * x + 8 * g + 4 * ln.hh;
            store4(dkr + d, make_float4(dk[x][4 * g], dk[x][4 * g + 1], dk[x][4 * g + 2], dk[x][4 * g + 3]),
                   (G.accumulate & PA_ACC_DK) != 0);
            float4 e = make_float4(dv[x][4 * g], dv[x][4 * g + 1], dv[x][4 * g + 2], dv[x][4 * g + 3]);
            if (mr) {
                const float4 m4 = *reinterpret_cast<const float4*>(mr + d);
                const float4 v4 = *reinterpret_cast<const float4*>(vr + d);
                store4(dmr + d, make_float4(e.x * v4.x, e.y * v4.y, e.z * v4.z, e.w * v4.w),
                       (G.accumulate & PA_ACC_DVMUL) != 0);
                e = make_float4(e.x * m4.x, e.y * m4.y, e.z * m4.z, e.w * m4.w);
            }
            store4(dvr + d, e, (G.accumulate & PA_ACC_DV) != 0);
        }
    if (ln.hh == 0 && G.dbias.ok()) {
        float* o = G.dbias.wrow<float>(b, h0, kj);
        *o = dbias + ((G.accumulate & PA_ACC_DBIAS) ? *o : 0.f);
    }
}

bool mfma_bwd_f32_supported(const GradDev& G) {
    const PassDev& P = G.f;
    if (P.dim != 64 && P.dim != 128) return false;
    if (P.km.p || P.qm.p || (P.flags & PA_FLAG_MAY_DEGENERATE)) return false;
    for (const DView* v : {&P.q, &P.k, &P.v, &G.dout, &G.dq, &G.dk, &G.dv})
        if (!aligned_rows_host(*v, 4)) return false;
    if (P.vmul.ok() && (!aligned_rows_host(P.vmul, 4) || !aligned_rows_host(G.dvmul, 4))) return false;
    return true;
}

// Row blocks per workgroup (R, sharing the staging and the splitting of the tiles) and waves per row
// block (C = 8 / R; head dim 128: 4 / R, its split operands need a SIMD's registers for one
// wave): the most row blocks that still give 256 workgroups, or 512 in causal grids, whose
// workgroups differ in length.  Forward, d = 64, N = 1024, us at R = 2 / 4 / 8: 4 x 16 heads causal
// 98 / 73 / 92, 8 x 16 heads 293 / - / 199, 4 x 8 heads causal 53 / 58 / 91, not causal 80 / 64 / 95.
static int f32_rows(int64_t units, int n, int dim, bool causal) {
    int r = dim == 64 ? 8 : 4;
    while (r > 2 && units * ((n + 32 * r - 1) / (32 * r)) < (causal ? 512 : 256)) r >>= 1;
    return r;
}

#define PA_F32_LAUNCH(KERN, ROWS, N, UNITS, ARG)                                                       \
    do {                                                                                              \
        const int r_ = (ROWS);                                                                        \
        const dim3 grid_((uint32_t)((UNITS) * (((N) + 32 * r_ - 1) / (32 * r_))));                     \
        if (P.dim == 64) {                                                                            \
            if (r_ == 8) hipLaunchKernelGGL((KERN<64, 8, 1>), grid_, dim3(512), 0, s, ARG);           \
            else if (r_ == 4) hipLaunchKernelGGL((KERN<64, 4, 2>), grid_, dim3(512), 0, s, ARG);      \
            else hipLaunchKernelGGL((KERN<64, 2, 4>), grid_, dim3(512), 0, s, ARG);                   \
        } else {                                                                                      \
            if (r_ == 4) hipLaunchKernelGGL((KERN<128, 4, 1>), grid_, dim3(256), 0, s, ARG);          \
            else hipLaunchKernelGGL((KERN<128, 2, 2>), grid_, dim3(256), 0, s, ARG);                  \
        }                                                                                             \
    } while (0)

// the profile's name of a launch: "split" where several waves share a row block
static bool f32_split(int rows, int dim) { return rows < (dim == 64 ? 8 : 4); }

void launch_mfma_bwd_f32(const GradDev& G, hipStream_t s) {
    const PassDev& P = G.f;
    // (unit counts in 64 bits: a product past 2^31 must not wrap into the small-grid test)
    const int64_t qunits = (int64_t)P.batch * P.heads, kunits = (int64_t)P.batch * G.hk;
    const int64_t qblocks = qunits * ((P.nq + 31) / 32);
    if (mfma_f32_block_applies(P, qblocks)) {
        launch_mfma_bwd_f32_dq_block(G, qblocks, s);
    } else {
        const int r = f32_rows(qunits, P.nq, P.dim, P.causal != 0);
        ProfScope ps(f32_split(r, P.dim) ? "mfma_bwd_f32_dq_split" : "mfma_bwd_f32_dq", s);
        PA_F32_LAUNCH(k_mfma_bwd_f32_dq, r, P.nq, qunits, G);
    }
    {
        const int r = f32_rows(kunits, P.nk, P.dim, P.causal != 0);
        ProfScope ps(f32_split(r, P.dim) ? "mfma_bwd_f32_dkv_split" : "mfma_bwd_f32_dkv", s);
        PA_F32_LAUNCH(k_mfma_bwd_f32_dkv, r, P.nk, kunits, G);
    }
}

bool mfma_fwd_f32_supported(const PassDev& P) {
    if (P.dim != 64 && P.dim != 128) return false;
    for (const DView* v : {&P.q, &P.k, &P.v, &P.out})
        if (!aligned_rows_host(*v, 4)) return false;
    if (P.vmul.ok() && !aligned_rows_host(P.vmul, 4)) return false;
    return true;
}

void launch_mfma_fwd_f32(const PassDev& P, hipStream_t s) {
    const int64_t units = (int64_t)P.batch * P.heads, blocks = units * ((P.nq + 31) / 32);
    if (mfma_f32_block_applies(P, blocks)) {
        launch_mfma_fwd_f32_block(P, blocks, s);
        return;
    }
    const int r = f32_rows(units, P.nq, P.dim, P.causal != 0);
    ProfScope ps(f32_split(r, P.dim) ? "mfma_fwd_f32_split" : "mfma_fwd_f32", s);
    PA_F32_LAUNCH(k_mfma_fwd_f32, r, P.nq, units, P);
}

}  // namespace pa
