// pa_mfma_f32.hip -- fp32 attention passes on the bf16 matrix cores (gfx950), head dim 64 or 128: the
// forward (every pass feature), and the backward of unmasked passes.
//
// Every fp32 operand is split into three bf16 numbers, x = h + m + l (each the rounding of what the
// ones before it leave: 8 + 8 + 8 significant bits, exact for all but the smallest numbers), and a
// product x y is the six of the nine partial products above 2^-26 of it: h h, h m, m h, m m, h l,
// l h, summed small ones first into the fp32 accumulators of v_mfma_f32_32x32x16_bf16.  That is 6
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
// gives. (A branch in each tile instead cost the backward kernels up to 200 spilled registers.)
// Masks, key bias classes, value multiplier, softclamp, causal limits and
// the module epilogue follow the pass semantics of polyattn.h; rows left fully masked get lse = NaN
// for k_fwd_fixup, as in the 16-bit kernels.
#include <algorithm>
#include <type_traits>

#include "pa_common.h"
#include "pa_launch.h"
#include "pa_mfma.h"

namespace pa {

constexpr int kF32BN = 32;             // rows per tile
constexpr float kF32Split = 3.38e38f;  // magnitudes above this do not split (bf16 would round to inf)

typedef Mma<bf16> MB;
typedef MB::frag bfrag;

// the three bf16 parts of 8 consecutive floats
struct Split8 {
    u32x4_t h, m, l;
    __device__ __forceinline__ bfrag fh() const { return __builtin_bit_cast(bfrag, h); }
    __device__ __forceinline__ bfrag fm() const { return __builtin_bit_cast(bfrag, m); }
    __device__ __forceinline__ bfrag fl() const { return __builtin_bit_cast(bfrag, l); }
};

__device__ __forceinline__ float bf_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

// `big`: some of them may exceed kF32Split (h is then truncated: exact residuals, no overflow)
__device__ __forceinline__ Split8 split8(const float (&x)[8], bool big = false) {
    Split8 s;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float a = x[2 * k], b = x[2 * k + 1];
        uint32_t h = pack2<bf16>(a, b);
        float ra = a - bf_lo(h), rb = b - bf_hi(h);
        if (big) {
            const uint32_t ua = __float_as_uint(a), ub = __float_as_uint(b);
            if (fabsf(a) > kF32Split) {
                h = (h & 0xffff0000u) | (ua >> 16);
                ra = fabsf(a) == INFINITY ? 0.f : a - __uint_as_float(ua & 0xffff0000u);
            }
            if (fabsf(b) > kF32Split) {
                h = (h & 0xffffu) | (ub & 0xffff0000u);
                rb = fabsf(b) == INFINITY ? 0.f : b - __uint_as_float(ub & 0xffff0000u);
            }
        }
        const uint32_t m = pack2<bf16>(ra, rb);
        s.h[k] = h;
        s.m[k] = m;
        s.l[k] = pack2<bf16>(ra - bf_lo(m), rb - bf_hi(m));
    }
    return s;
}

__device__ __forceinline__ float max_abs8(const float (&x)[8], float mx) {
#pragma unroll
    for (int e = 0; e < 8; e += 2) mx = fmaxf(fmaxf(mx, fabsf(x[e])), fabsf(x[e + 1]));
    return mx;
}

// a fragment with its infinities and NaNs as zeros
__device__ __forceinline__ bfrag finite(bfrag f) {
    u32x4_t w = __builtin_bit_cast(u32x4_t, f);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if ((w[k] & 0x7f80u) == 0x7f80u) w[k] &= 0xffff0000u;
        if ((w[k] & 0x7f800000u) == 0x7f800000u) w[k] &= 0xffffu;
    }
    return __builtin_bit_cast(bfrag, w);
}

// the five small partial products, smallest first (BIG: some h may be infinite)
template <bool BIG>
__device__ __forceinline__ f32x16_t mma_small(bfrag ah, bfrag am, bfrag al, const Split8& b, f32x16_t c) {
    bfrag bh = b.fh();
    if (BIG) {
        ah = finite(ah);
        bh = finite(bh);
    }
    c = MB::run(al, bh, c);
    c = MB::run(ah, b.fl(), c);
    c = MB::run(am, b.fm(), c);
    c = MB::run(am, bh, c);
    return MB::run(ah, b.fm(), c);
}

// One 32-row tile of a tensor in LDS: planes h, m, l of [32][D] bf16, 16-byte chunks swizzled.
template <int D>
struct X3 {
    static constexpr int PLANE = kF32BN * D;  // elements
    static constexpr int TILE = 3 * PLANE;
    static constexpr int CPR = D / 8;

    // chunk permutation of a row, conflict-free for row fragments and transposed reads
    static __device__ __forceinline__ int swz(int r) {
        if (D == 64) {
            const int v = (r >> 1) & 7;
            return ((v & 1) << 2) | (v & 2) | ((v >> 2) & 1);
        }
        const int v = r & 15;
        return ((v & 1) << 3) | ((v & 2) << 1) | ((v >> 1) & 2) | ((v >> 3) & 1);
    }
    static __device__ __forceinline__ void store(bf16* t, int r, int ch, const Split8& s) {
        bf16* p = t + r * D + ((ch ^ swz(r)) * 8);
        *reinterpret_cast<u32x4_t*>(p) = s.h;
        *reinterpret_cast<u32x4_t*>(p + PLANE) = s.m;
        *reinterpret_cast<u32x4_t*>(p + 2 * PLANE) = s.l;
    }
};

// Per-lane LDS offsets of a tile's operands: row fragments (row l % 32, features 16c + 8 hh ..)
// and transposed ones (rows 16 t2 + .., features 32x + l % 32).
template <int D>
struct X3Lane {
    using L = X3<D>;
    int col, hh;
    int toff[2][D / 32];
    __device__ __forceinline__ void init(int lane) {
        col = lane & 31;
        hh = lane >> 5;
        const int g = lane >> 4, j = lane & 15;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int r = 8 * u + 4 * (g >> 1) + (j >> 2);
#pragma unroll
            for (int x = 0; x < D / 32; ++x) {
                const int ch = 4 * x + 2 * (g & 1) + ((j & 3) >> 1);
                toff[u][x] = r * D + ((ch ^ L::swz(r)) * 8) + 4 * (j & 1);
            }
        }
    }
    __device__ __forceinline__ bfrag row(const bf16* t, int plane, int c) const {
        return ld_frag<bf16>(t + plane * L::PLANE + col * D + (((2 * c + hh) ^ L::swz(col)) * 8));
    }
    // (the swizzle depends on the row modulo 16 only)
    __device__ __forceinline__ bfrag tr(const bf16* t, int plane, int t2, int x) const {
        const bf16* p = t + plane * L::PLANE + 16 * t2 * D;
        const u32x2_t lo = lds_read_tr(p + toff[0][x]), hi = lds_read_tr(p + toff[1][x]);
        const u32x4_t v = {lo[0], lo[1], hi[0], hi[1]};
        return __builtin_bit_cast(bfrag, v);
    }
    // s += T B: T the tile's rows, B the wave's 32 split rows (lane = column)
    template <bool BIG>
    __device__ __forceinline__ void rows_mma(const bf16* t, const Split8 (&b)[D / 16], f32x16_t& s) const {
#pragma unroll
        for (int c = 0; c < D / 16; ++c) s = mma_small<BIG>(row(t, 0, c), row(t, 1, c), row(t, 2, c), b[c], s);
#pragma unroll
        for (int c = 0; c < D / 16; ++c) s = MB::run(row(t, 0, c), b[c].fh(), s);
    }
    // o += T^T P: P the score registers p (rows of the tile x the wave's columns)
    template <bool BIG>
    __device__ __forceinline__ void cols_mma(const bf16* t, const f32x16_t& p, f32x16_t (&o)[D / 32]) const {
#pragma unroll
        for (int t2 = 0; t2 < 2; ++t2) {
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = p[8 * t2 + e];
            const Split8 b = split8(v, BIG);
#pragma unroll
            for (int x = 0; x < D / 32; ++x) {
                const bfrag ah = tr(t, 0, t2, x);
                o[x] = MB::run(ah, b.fh(), mma_small<BIG>(ah, tr(t, 1, t2, x), tr(t, 2, t2, x), b, o[x]));
            }
        }
    }
};

// The wave's 32 rows of a tensor (times a multiplier's) as split B operands; returns whether some
// value does not split (uniform).
template <int D, bool BIG>
__device__ __forceinline__ bool x3_load_rows(const float* row, const float* mul, bool ok, int hh,
                                             Split8 (&f)[D / 16]) {
    float v[D / 16][8];
    float mx = 0.f;
#pragma unroll
    for (int c = 0; c < D / 16; ++c) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            float4 a = *reinterpret_cast<const float4*>(row + 16 * c + 8 * hh + 4 * q);
            if (mul) {
                const float4 m = *reinterpret_cast<const float4*>(mul + 16 * c + 8 * hh + 4 * q);
                a = make_float4(a.x * m.x, a.y * m.y, a.z * m.z, a.w * m.w);
            }
            v[c][4 * q] = ok ? a.x : 0.f;
            v[c][4 * q + 1] = ok ? a.y : 0.f;
            v[c][4 * q + 2] = ok ? a.z : 0.f;
            v[c][4 * q + 3] = ok ? a.w : 0.f;
        }
        mx = max_abs8(v[c], mx);
    }
#pragma unroll
    for (int c = 0; c < D / 16; ++c) f[c] = split8(v[c], BIG);
    return __any(mx > kF32Split);
}

// Whether some thread of the workgroup met a value that does not split (every thread calls it).
__device__ __forceinline__ bool x3_met_big(float mx, int* flag) {
    __syncthreads();
    if (threadIdx.x == 0) *flag = 0;
    __syncthreads();
    if (mx > kF32Split) *flag = 1;
    __syncthreads();
    return *flag != 0;
}

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

__device__ __forceinline__ float key_term_l2(const PassDev& P, int b, int h, int j) {
    if (j >= P.nk) return -INFINITY;
    const float x = P.bias.ok() ? P.bias.scalar(b, h, j) : 0.f;
    return bias_class(x) == 0 ? x * kLog2e : -INFINITY;
}

// one 4-element group of an output row: value (+ the old value with accumulate)
__device__ __forceinline__ void store4(float* p, float4 v, bool acc) {
    if (acc) {
        const float4 o = *reinterpret_cast<const float4*>(p);
        v.x += o.x;
        v.y += o.y;
        v.z += o.z;
        v.w += o.w;
    }
    *reinterpret_cast<float4*>(p) = v;
}

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
                float mx[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
                for (int i = 0; i < 16; ++i) s[i] *= P.scale;
                if (sc) {
                    keep_branch();
#pragma unroll
                    for (int i = 0; i < 16; ++i) s[i] = softclamp_f(s[i], P.softclamp);
                }
#pragma unroll
                for (int g = 0; g < 4; ++g) {  // one rounding, as in the backward
                    const float4 bb = *reinterpret_cast<const float4*>(B + 8 * g + 4 * ln.hh);
                    s[4 * g] = fmaf(s[4 * g], kLog2e, bb.x);
                    s[4 * g + 1] = fmaf(s[4 * g + 1], kLog2e, bb.y);
                    s[4 * g + 2] = fmaf(s[4 * g + 2], kLog2e, bb.z);
                    s[4 * g + 3] = fmaf(s[4 * g + 3], kLog2e, bb.w);
                }
                if (causal && j0 + 31 > q0) {
                    keep_branch();
                    const int lim = qi - j0 - 4 * ln.hh;
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        if (8 * (i / 4) + (i % 4) > lim) s[i] = -INFINITY;
                }
#pragma unroll
                for (int i = 0; i < 16; ++i) mx[i % 4] = fmaxf(mx[i % 4], s[i]);
                const float mnew = fmaxf(m, xhalf_max(fmaxf(fmaxf(mx[0], mx[1]), fmaxf(mx[2], mx[3]))));
                if (__any(mnew > m)) {
                    keep_branch();
                    const float a = mnew > m ? (m == -INFINITY ? 0.f : fast_exp2(m - mnew)) : 1.f;
                    l *= a;
#pragma unroll
                    for (int x = 0; x < D / 32; ++x)
#pragma unroll
                        for (int i = 0; i < 16; ++i) o[x][i] *= a;
                    m = mnew;
                }
                const float msub = m == -INFINITY ? 0.f : m;  // (nothing but -inf scores yet: p = 0)
                float lt[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    s[i] = fast_exp2(s[i] - msub);
                    lt[i % 4] += s[i];
                }
                l += (lt[0] + lt[1]) + (lt[2] + lt[3]);
                ln.template cols_mma<BIG>(V, s, o);
            }
        }
    };
    sweep(std::false_type());
    if (__builtin_expect(x3_met_big(big, &sF), 0)) sweep(std::true_type());
    if (C > 1) {
        // the C softmax states of a row block, merged by its first wave
        float* buf = reinterpret_cast<float*>(sT);
        __syncthreads();
        if (wc > 0) {
            float* so = buf + ((wr * (C - 1) + wc - 1) * (NO + 2)) * 64 + lane;
#pragma unroll
            for (int x = 0; x < D / 32; ++x)
#pragma unroll
                for (int i = 0; i < 16; ++i) so[(x * 16 + i) * 64] = o[x][i];
            so[NO * 64] = m;
            so[(NO + 1) * 64] = l;
        }
        __syncthreads();
        if (wc != 0) return;  // no barriers below
        float mt = m;
#pragma unroll
        for (int v = 0; v < C - 1; ++v) mt = fmaxf(mt, buf[((wr * (C - 1) + v) * (NO + 2) + NO) * 64 + lane]);
        const float a0 = m == -INFINITY ? 0.f : fast_exp2(m - mt);
        l *= a0;
#pragma unroll
        for (int x = 0; x < D / 32; ++x)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[x][i] *= a0;
#pragma unroll
        for (int v = 0; v < C - 1; ++v) {
            const float* so = buf + ((wr * (C - 1) + v) * (NO + 2)) * 64 + lane;
            const float mv = so[NO * 64], a = mv == -INFINITY ? 0.f : fast_exp2(mv - mt);
            l += so[(NO + 1) * 64] * a;
#pragma unroll
            for (int x = 0; x < D / 32; ++x)
#pragma unroll
                for (int i = 0; i < 16; ++i) o[x][i] += so[(x * 16 + i) * 64] * a;
        }
        m = mt;
    }

    // the outputs, lse (NaN for a row left fully masked, for k_fwd_fixup) and the module epilogue
    const float lt = xhalf_sum(l);
    if (qi >= P.nq) return;
    const bool degenerate = !(lt > 0.f) || !P.qm.keep(b, qi);
    const float inv = degenerate ? 0.f : 1.f / lt;
    float* orow = P.out.wrow<float>(b, h, qi);
#pragma unroll
    for (int x = 0; x < D / 32; ++x)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int d = 32 * x + 8 * g + 4 * ln.hh;
            const float4 v = make_float4(o[x][4 * g] * inv, o[x][4 * g + 1] * inv,
                                         o[x][4 * g + 2] * inv, o[x][4 * g + 3] * inv);
            *reinterpret_cast<float4*>(orow + d) = v;
            if (P.ey.ok()) {
                float* yrow = P.ey.wrow<float>(b, h, qi);
                yrow[d] = epi_y<float>(P, b, h, qi, d, v.x);
                yrow[d + 1] = epi_y<float>(P, b, h, qi, d + 1, v.y);
                yrow[d + 2] = epi_y<float>(P, b, h, qi, d + 2, v.z);
                yrow[d + 3] = epi_y<float>(P, b, h, qi, d + 3, v.w);
            }
        }
    if (ln.hh == 0) *P.lse.wrow<float>(b, h, qi) = degenerate ? NAN : (m + log2f(lt)) * kLn2;
}

// ---------------------------------------------------------------------------------------
// backward (unmasked passes; after the row preprocess: ws_lse, ws_D)

// the largest of mx and the block's magnitudes (dS of overflowing gradients may not split)
__device__ __forceinline__ float max_abs16(const f32x16_t& s, float mx) {
#pragma unroll
    for (int i = 0; i < 16; i += 2) mx = fmaxf(fmaxf(mx, fabsf(s[i])), fabsf(s[i + 1]));
    return mx;
}

// The C partial sums of a row block added into its first wave's registers, in wave order;
// returns true in the waves that are then done.
template <int NB, int R, int C>
__device__ __forceinline__ bool x3_merge(f32x16_t* const (&acc)[NB], float* extra, float* buf, int wr,
                                         int wc, int lane) {
    if (C == 1) return false;
    constexpr int ST = (NB * 16 + 1) * 64;
    __syncthreads();
    if (wc > 0) {
        float* so = buf + (wr * (C - 1) + wc - 1) * ST + lane;
#pragma unroll
        for (int x = 0; x < NB; ++x)
#pragma unroll
            for (int i = 0; i < 16; ++i) so[(x * 16 + i) * 64] = (*acc[x])[i];
        so[NB * 16 * 64] = *extra;
    }
    __syncthreads();
    if (wc != 0) return true;
#pragma unroll
    for (int v = 0; v < C - 1; ++v) {
        const float* so = buf + (wr * (C - 1) + v) * ST + lane;
#pragma unroll
        for (int x = 0; x < NB; ++x)
#pragma unroll
            for (int i = 0; i < 16; ++i) (*acc[x])[i] += so[(x * 16 + i) * 64];
        *extra += so[NB * 16 * 64];
    }
    return false;
}

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
            const int lim = causal ? qi - j0 - 4 * ln.hh : 1 << 30;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const float4 bb = *reinterpret_cast<const float4*>(B + 8 * g + 4 * ln.hh);
                const float bv[4] = {bb.x, bb.y, bb.z, bb.w};
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int i = 4 * g + k;
                    float y = s[i] * P.scale;
                    if (sc) y = softclamp_f(y, P.softclamp);
                    float t = y * kLog2e + bv[k];
                    if (8 * g + k > lim) t = -INFINITY;
                    const float p = fast_exp2(t - lse_l2);
                    float ds = p * (dp[i] - dsum);
                    if (sc) ds *= softclamp_grad(y, P.softclamp);
                    s[i] = ds * P.scale;
                }
            }
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
    if (!qrow) return;
    float* row = G.dq.wrow<float>(b, h, qi);
    const bool acc = (G.accumulate & PA_ACC_DQ) != 0;
#pragma unroll
    for (int x = 0; x < D / 32; ++x)
#pragma unroll
        for (int g = 0; g < 4; ++g)
            store4(row + 32 * x + 8 * g + 4 * ln.hh,
                   make_float4(dq[x][4 * g], dq[x][4 * g + 1], dq[x][4 * g + 2], dq[x][4 * g + 3]), acc);
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
    {
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
    const int64_t units = (int64_t)P.batch * P.heads;
    const int r = f32_rows(units, P.nq, P.dim, P.causal != 0);
    ProfScope ps(f32_split(r, P.dim) ? "mfma_fwd_f32_split" : "mfma_fwd_f32", s);
    PA_F32_LAUNCH(k_mfma_fwd_f32, r, P.nq, units, P);
}

}  // namespace pa
