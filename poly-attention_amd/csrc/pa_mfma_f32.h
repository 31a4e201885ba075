// pa_mfma_f32.h -- pieces of the fp32 attention passes on the bf16 matrix cores that their kernels share
// (pa_mfma_f32.hip, where the method is described, and pa_mfma_f32_block.hip).
#pragma once

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

// The softmax update of one key tile: raw scores s -> probabilities against the running max m (log2
// units, shared by the lane pair), o and l rescaled, l the lane's partial sum.  B: the tile's key
// terms; with `cut`, keys after position lim of the lane's rows are masked.
template <int D>
__device__ __forceinline__ void f32_softmax_tile(const PassDev& P, f32x16_t& s, const float* B, bool sc,
                                                 bool cut, int lim, int hh, f32x16_t (&o)[D / 32],
                                                 float& m, float& l) {
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
        const float4 bb = *reinterpret_cast<const float4*>(B + 8 * g + 4 * hh);
        s[4 * g] = fmaf(s[4 * g], kLog2e, bb.x);
        s[4 * g + 1] = fmaf(s[4 * g + 1], kLog2e, bb.y);
        s[4 * g + 2] = fmaf(s[4 * g + 2], kLog2e, bb.z);
        s[4 * g + 3] = fmaf(s[4 * g + 3], kLog2e, bb.w);
    }
    if (cut) {
        keep_branch();
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
}

// The C softmax states of a row block merged by its first wave; returns true in the others, which
// are then done.
template <int D, int R, int C>
__device__ __forceinline__ bool x3_merge_softmax(f32x16_t (&o)[D / 32], float& m, float& l, float* buf, int wr,
                                                 int wc, int lane) {
    if (C == 1) return false;
    constexpr int NO = D / 32 * 16;
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
    if (wc != 0) return true;
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
    return false;
}

// a query row's output from its softmax state, lse (NaN for a row left fully masked, for
// k_fwd_fixup) and the module epilogue
template <int D>
__device__ __forceinline__ void f32_store_out(const PassDev& P, int b, int h, int qi, int hh,
                                              const f32x16_t (&o)[D / 32], float m, float l) {
    const float lt = xhalf_sum(l);
    if (qi >= P.nq) return;
    const bool degenerate = !(lt > 0.f) || !P.qm.keep(b, qi);
    const float inv = degenerate ? 0.f : 1.f / lt;
    float* orow = P.out.wrow<float>(b, h, qi);
#pragma unroll
    for (int x = 0; x < D / 32; ++x)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int d = 32 * x + 8 * g + 4 * hh;
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
    if (hh == 0) *P.lse.wrow<float>(b, h, qi) = degenerate ? NAN : (m + log2f(lt)) * kLn2;
}

// ---------------------------------------------------------------------------------------
// backward

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

// A query-major tile's dS * scale in s, from the raw scores s and dP (lane = query; keys after
// position lim of the lane's rows masked).
template <int D>
__device__ __forceinline__ void f32_ds_query(const PassDev& P, f32x16_t& s, const f32x16_t& dp, const float* B,
                                             bool sc, int lim, int hh, float lse_l2, float dsum) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const float4 bb = *reinterpret_cast<const float4*>(B + 8 * g + 4 * hh);
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
}

template <int D>
__device__ __forceinline__ void f32_store_dq(const GradDev& G, int b, int h, int qi, int hh,
                                             const f32x16_t (&dq)[D / 32]) {
    float* row = G.dq.wrow<float>(b, h, qi);
    const bool acc = (G.accumulate & PA_ACC_DQ) != 0;
#pragma unroll
    for (int x = 0; x < D / 32; ++x)
#pragma unroll
        for (int g = 0; g < 4; ++g)
            store4(row + 32 * x + 8 * g + 4 * hh,
                   make_float4(dq[x][4 * g], dq[x][4 * g + 1], dq[x][4 * g + 2], dq[x][4 * g + 3]), acc);
}

}  // namespace pa
