// pa_norm.hip -- row RMSNorm over the head dim of [batch, heads, n, dim] views (the q/k norms
// of the poly-attention modules), optionally followed by the rotary embedding, forward and
// backward.  HBM bound: a row group of LPR lanes
// reads a whole row with 16-byte loads, reduces with DPP inside the row group, and writes the
// row back; the backward writes dx and accumulates the weight gradient per workgroup into a
// fixed partial row, summed afterwards in a fixed order (deterministic, no atomics).
#include <algorithm>
#include <type_traits>

#include "pa_common.h"
#include "pa_launch.h"

namespace pa {

// n / d for n < 2^31 by a multiply-high and a shift (d fixed per launch; l = ceil(log2 d),
// m = floor(2^32 (2^l - d) / d) + 1)
struct FastDiv {
    uint32_t d, m, l;
    __device__ __forceinline__ uint32_t div(uint32_t n) const { return (__umulhi(m, n) + n) >> l; }
};
static FastDiv make_fastdiv(uint32_t d) {
    uint32_t l = 0;
    while ((1ull << l) < d) ++l;
    FastDiv f;
    f.d = d;
    f.l = l;
    f.m = (uint32_t)((((1ull << 32) * ((1ull << l) - d)) / d) + 1);
    return f;
}

constexpr int kRmsThreads = 256;
constexpr int kRmsMaxBlocks = 1024;
constexpr int kRmsU = 4;  // rows per row group and pass

// a strided [batch, heads, n, dim] tensor as the norm kernels address it (element strides)
struct RView {
    char* p;
    int64_t sb, sh, sn;
    template <typename T> __device__ __forceinline__ T* at(uint32_t b, uint32_t h, uint32_t i) const {
        return reinterpret_cast<T*>(p) + ((int64_t)b * sb + (int64_t)h * sh + (int64_t)i * sn);
    }
};

struct RmsDev {
    int32_t batch, heads, n, dim, lpr;
    int32_t hfast;    // rows walk heads fastest (input laid out [B, N, H, dim])
    uint32_t rows;    // < 2^31 (checked on the host)
    FastDiv fd_n, fd_h;
    float eps, inv_dim;
    RView x, y, dy, dx;
    const void* w;
    int32_t wdt;
    float* rstd;      // [batch][heads][n]
    float* partial;   // [gridDim.x][dim] (backward)
    float* dw;        // [dim] (backward, fp32)
    const void* ang;  // rotary angles [n][astride] or null
    int32_t adt, rot_dim;
    int64_t astride;
    int32_t trig;     // slots of a run's cos / sin table (0: evaluated per row)
};


template <typename T> struct RVec;
template <> struct RVec<bf16> { static constexpr int n = 8; };
template <> struct RVec<f16> { static constexpr int n = 8; };
template <> struct RVec<float> { static constexpr int n = 4; };

template <int LPR>
__device__ __forceinline__ float row_sum(float x) {
#pragma unroll
    for (int off = 1; off < LPR; off <<= 1) x += __shfl_xor(x, off);
    return x;
}

template <typename T>
__device__ __forceinline__ void load_row(const T* p, bool ok, float* out) {
    constexpr int E = RVec<T>::n;
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    u32x4 raw = {0u, 0u, 0u, 0u};
    if (ok) raw = *reinterpret_cast<const u32x4*>(p);
    const T* e = reinterpret_cast<const T*>(&raw);
#pragma unroll
    for (int i = 0; i < E; ++i) out[i] = to_f(e[i]);
}

template <typename T>
__device__ __forceinline__ void store_row(T* p, const float* v) {
    constexpr int E = RVec<T>::n;
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    u32x4 raw;
    T* e = reinterpret_cast<T*>(&raw);
#pragma unroll
    for (int i = 0; i < E; ++i) e[i] = from_f<T>(v[i]);
    *reinterpret_cast<u32x4*>(p) = raw;
}

// cos and sin of the rotary angles, once per position instead of once per row (full-range cosf / sinf
// of 8 features were half the time of the rotary kernels): where rows walk heads fastest, the
// RPB consecutive rows of a run span few positions, and a workgroup first fills a table of theirs
// in LDS, for each of the kRmsU runs of its next pass.  The same functions of the same angles, so
// the results are the same bits.  B = 2, H = 16, N = 2048, d = 64, bf16: forward 18.7 -> 12.6 us,
// backward 22.8 -> 14.0 us.
constexpr int kTrigMax = 3072;  // entries (24 KB)

__device__ __forceinline__ float2 rope_trig(const RmsDev& R, uint32_t pos, int d) {
    const float a = load_any(R.ang, R.adt, (int64_t)pos * R.astride + d);
    return make_float2(cosf(a), sinf(a));
}

// the kRmsU runs of rows [first + u step, + rpb): slot k of run u holds position (token / heads + k)
// modulo n (every thread calls it; ends with a barrier)
__device__ __forceinline__ void fill_trig(const RmsDev& R, float2* tab, uint32_t first, uint32_t step) {
    __syncthreads();  // the previous pass has read its table
    const int per = R.trig * R.rot_dim;
    for (int e = threadIdx.x; e < kRmsU * per; e += kRmsThreads) {
        const int u = e / per, k = (e % per) / R.rot_dim, d = e % R.rot_dim;
        const uint32_t r = first + u * step;
        const uint32_t tok = R.fd_h.div(r < R.rows ? r : 0u) + k;
        tab[e] = rope_trig(R, tok - R.fd_n.div(tok) * R.fd_n.d, d);
    }
    __syncthreads();
}

// where a kernel's rotation takes its cos / sin from: a template argument, since the code of both ways
// and the table's LDS cost the norms without a table (fewer than 4 heads, contiguous heads) up to
// 45%: 4 x 16 heads x 4096, d = 64, bf16, contiguous, forward 42 us before the table, 61 with both
// ways in one kernel, 44 like this; 2 heads x 512 12.2, 15.0 and 13.0.
enum { kRopeNone, kRopeRows, kRopeTable, kRopeEither };  // either: by R.trig

template <int ROPE>
__device__ __forceinline__ bool rope_table(const RmsDev& R) {
    return ROPE == kRopeTable || (ROPE == kRopeEither && R.trig);
}

// f(get), get(e) the cos / sin of feature d0 + e of row r (of the run starting at `first`, in slot row
// u): all read from the table, or evaluated, at once; with PAIRS evaluated as they are used (the
// forward's array of eight took it from 119 to 135 registers; the 16-bit backward, three waves a
// SIMD either way, is 5% faster with it)
template <int ROPE, int E, bool PAIRS, class F>
__device__ __forceinline__ void with_trig(const RmsDev& R, const float2* tab, int u, uint32_t first,
                                          uint32_t r, uint32_t pos, int d0, F f) {
    float2 t[E];
    if (rope_table<ROPE>(R)) {
        const int k = (int)(R.fd_h.div(r) - R.fd_h.div(first));
        const float2* p = tab + (u * R.trig + k) * R.rot_dim + d0;
#pragma unroll
        for (int e = 0; e < E; ++e)
            if (d0 + e < R.rot_dim) t[e] = p[e];
    } else if (PAIRS) {
        f([&](int e) __attribute__((always_inline)) { return rope_trig(R, pos, d0 + e); });
        return;
    } else {
#pragma unroll
        for (int e = 0; e < E; ++e)
            if (d0 + e < R.rot_dim) t[e] = rope_trig(R, pos, d0 + e);
    }
    f([&](int e) __attribute__((always_inline)) { return t[e]; });
}

// a result in fp32 of its own.  Every kernel of the norms gives the same bits: sums of products are
// written as the fused operations that they are, and an fp16 conversion is not fused into one (a
// compiler does that where no branch lies between).
template <typename T>
__device__ __forceinline__ float own(float x) {
    if (std::is_same<T, f16>::value) asm("" : "+v"(x));
    return x;
}

// rotary embedding of the E features d0.. of one row in place (fp32 math on the rounded
// norm output t, one rounding when stored): y[2i] = t[2i] cos a[2i] - t[2i+1] sin a[2i],
// y[2i+1] = t[2i+1] cos a[2i+1] + t[2i] sin a[2i+1]
template <typename T, int E, class Get>
__device__ __forceinline__ void rope_fwd(const RmsDev& R, int d0, Get get, float (&t)[E]) {
#pragma unroll
    for (int e = 0; e < E; e += 2) {
        if (d0 + e >= R.rot_dim) break;
        const float2 a = get(e), b = get(e + 1);
        const float t0 = t[e], t1 = t[e + 1];
        t[e] = own<T>(fmaf(t0, a.x, -(t1 * a.y)));
        t[e + 1] = own<T>(fmaf(t1, b.x, t0 * b.y));
    }
}

// the gradient of t from the gradient g of the rotated row (the transposed rotation)
template <typename T, int E, class Get>
__device__ __forceinline__ void rope_bwd(const RmsDev& R, int d0, Get get, float (&g)[E]) {
#pragma unroll
    for (int e = 0; e < E; e += 2) {
        if (d0 + e >= R.rot_dim) break;
        const float2 a = get(e), b = get(e + 1);
        const float g0 = g[e], g1 = g[e + 1];
        g[e] = own<T>(fmaf(g0, a.x, g1 * b.y));
        g[e + 1] = own<T>(fmaf(g1, b.x, -(g0 * a.y)));
    }
}

// row r -> (batch, head, position) in the order that walks the input's memory sequentially
__device__ __forceinline__ void row_coords(const RmsDev& R, uint32_t r, uint32_t& b, uint32_t& h,
                                           uint32_t& i) {
    if (R.hfast) {
        const uint32_t q1 = R.fd_h.div(r);
        h = r - q1 * R.fd_h.d;
        b = R.fd_n.div(q1);
        i = q1 - b * R.fd_n.d;
    } else {
        const uint32_t q1 = R.fd_n.div(r);
        i = r - q1 * R.fd_n.d;
        b = R.fd_h.div(q1);
        h = q1 - b * R.fd_h.d;
    }
}

__device__ __forceinline__ uint32_t rstd_index(const RmsDev& R, uint32_t b, uint32_t h, uint32_t i) {
    return (b * R.fd_h.d + h) * R.fd_n.d + i;
}

// y = round(x * rsqrt(mean(x^2) + eps) * w); rstd saved per row.  Each row group handles
// kRmsU rows per pass, their loads issued together (memory-level parallelism).
template <typename T, int LPR, int ROPE>
__device__ __forceinline__ void rms_fwd_rows(const RmsDev& R) {
    constexpr int E = RVec<T>::n;
    constexpr int RPB = kRmsThreads / LPR;  // row groups per block
    const int sub = threadIdx.x % LPR, rg = threadIdx.x / LPR;
    const int d0 = sub * E;
    const bool dok = d0 < R.dim;
    float w[E];
#pragma unroll
    for (int e = 0; e < E; ++e) w[e] = (R.w && dok) ? load_any(R.w, R.wdt, d0 + e) : 1.f;
    const uint32_t step = gridDim.x * RPB;
    __shared__ float2 tab[ROPE >= kRopeTable ? kTrigMax : 1];
    for (uint32_t first = blockIdx.x * RPB; first < R.rows; first += step * kRmsU) {
        const uint32_t r0 = first + rg;
        if (rope_table<ROPE>(R)) fill_trig(R, tab, first, step);
        float x[kRmsU][E];
        uint32_t b[kRmsU], h[kRmsU], i[kRmsU];
#pragma unroll
        for (int u = 0; u < kRmsU; ++u) {
            const uint32_t r = r0 + u * step;
            row_coords(R, r < R.rows ? r : 0u, b[u], h[u], i[u]);
            load_row<T>(R.x.at<T>(b[u], h[u], i[u]) + d0, dok && r < R.rows, x[u]);
        }
#pragma unroll
        for (int u = 0; u < kRmsU; ++u) {
            const uint32_t r = r0 + u * step;
            float ss = 0.f;
#pragma unroll
            for (int e = 0; e < E; ++e) ss += x[u][e] * x[u][e];
            ss = row_sum<LPR>(ss);
            if (r >= R.rows) continue;
            const float rs = rsqrtf(ss * R.inv_dim + R.eps);
            if (dok) {
                float y[E];
#pragma unroll
                for (int e = 0; e < E; ++e) y[e] = (x[u][e] * rs) * w[e];
                if (ROPE && d0 < R.rot_dim) {
                    // the norm output is a tensor of T before the rotation
#pragma unroll
                    for (int e = 0; e < E; ++e) y[e] = round_to<T>(y[e]);
                    with_trig<ROPE, E, true>(R, tab, u, first + u * step, r, i[u], d0,
                                             [&](auto get) __attribute__((always_inline)) { rope_fwd<T, E>(R, d0, get, y); });
                }
                store_row<T>(R.y.at<T>(b[u], h[u], i[u]) + d0, y);
            }
            if (sub == 0 && R.rstd) R.rstd[rstd_index(R, b[u], h[u], i[u])] = rs;
        }
    }
}

// (four waves per SIMD: 129 registers without the bound at LPR = 16 with rotary)
template <typename T, int LPR, int ROPE>
__global__ __launch_bounds__(kRmsThreads, 4) void k_rms_fwd(RmsDev R) {
    rms_fwd_rows<T, LPR, ROPE>(R);
}

// several norms in one launch (pa_rmsnorm_fwd_many, pa_rmsnorm_many): blockIdx.y selects the tensor.
// A norm of a layer is 5 to 15 us, as long as the host's part in its launch, so a layer's three or
// four norms go out together, backward and weight gradients too: training step of an order-3 layer
// (2 x 2048 x 1024, 16 heads) 1246 -> 1144 us, gated order-2 layer (4 x 1024 x 512) 1253 -> 1165 us.
struct RmsMany {
    RmsDev it[PA_RMS_MAX_ITEMS];
};

template <typename T, int LPR, int ROPE>
__global__ __launch_bounds__(kRmsThreads, 4) void k_rms_fwd_many(RmsMany M) {
    rms_fwd_rows<T, LPR, ROPE>(M.it[blockIdx.y]);
}

// dx = rstd * (g - xhat * mean(g * xhat)), g = dy * w, xhat = x * rstd; the block's weight
// gradient partial sum_rows dy * xhat goes to partial[blockIdx.x]
template <typename T, int LPR, int ROPE>
__device__ __forceinline__ void rms_bwd_rows(const RmsDev& R) {
    constexpr int E = RVec<T>::n;
    constexpr int RPB = kRmsThreads / LPR;
    __shared__ float s_dw[kRmsThreads / 64][512];
    const int sub = threadIdx.x % LPR, rg = threadIdx.x / LPR;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int d0 = sub * E;
    const bool dok = d0 < R.dim;
    float w[E], acc[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        w[e] = (R.w && dok) ? load_any(R.w, R.wdt, d0 + e) : 1.f;
        acc[e] = 0.f;
    }
    const uint32_t step = gridDim.x * RPB;
    __shared__ float2 tab[ROPE >= kRopeTable ? kTrigMax : 1];
    for (uint32_t first = blockIdx.x * RPB; first < R.rows; first += step * kRmsU) {
        const uint32_t r0 = first + rg;
        if (rope_table<ROPE>(R)) fill_trig(R, tab, first, step);
        float x[kRmsU][E], dy[kRmsU][E], rs[kRmsU];
        uint32_t b[kRmsU], h[kRmsU], i[kRmsU];
#pragma unroll
        for (int u = 0; u < kRmsU; ++u) {
            const uint32_t r = r0 + u * step;
            const bool ok = r < R.rows;
            row_coords(R, ok ? r : 0u, b[u], h[u], i[u]);
            load_row<T>(R.x.at<T>(b[u], h[u], i[u]) + d0, dok && ok, x[u]);
            load_row<T>(R.dy.at<T>(b[u], h[u], i[u]) + d0, dok && ok, dy[u]);
            rs[u] = ok ? R.rstd[rstd_index(R, b[u], h[u], i[u])] : 0.f;
        }
        if (ROPE && d0 < R.rot_dim) {
            // back through the rotation: the gradient of the norm output, a tensor of T
#pragma unroll
            for (int u = 0; u < kRmsU; ++u) {
                const uint32_t r = r0 + u * step;
                with_trig<ROPE, E, E == 4>(
                    R, tab, u, first + u * step, r < R.rows ? r : first + u * step, i[u], d0,
                    [&](auto get) __attribute__((always_inline)) { rope_bwd<T, E>(R, d0, get, dy[u]); });
#pragma unroll
                for (int e = 0; e < E; ++e) dy[u][e] = round_to<T>(dy[u][e]);
            }
        }
#pragma unroll
        for (int u = 0; u < kRmsU; ++u) {
            float c = 0.f;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const float xh = x[u][e] * rs[u];
                c = fmaf(dy[u][e] * w[e], xh, c);
                acc[e] = fmaf(dy[u][e], xh, acc[e]);
            }
            c = row_sum<LPR>(c) * R.inv_dim;
            if (r0 + u * step < R.rows && dok) {
                float dx[E];
#pragma unroll
                for (int e = 0; e < E; ++e) dx[e] = own<T>(rs[u] * fmaf(dy[u][e], w[e], -(x[u][e] * rs[u] * c)));
                store_row<T>(R.dx.at<T>(b[u], h[u], i[u]) + d0, dx);
            }
        }
    }
    if (!R.partial) return;
    // reduce acc over the row groups of the wave (lanes sub, sub + LPR, ...), then the waves
#pragma unroll
    for (int e = 0; e < E; ++e)
        for (int off = LPR; off < 64; off <<= 1) acc[e] += __shfl_xor(acc[e], off);
    if (lane < LPR && dok)
#pragma unroll
        for (int e = 0; e < E; ++e) s_dw[wave][d0 + e] = acc[e];
    __syncthreads();
    for (int f = threadIdx.x; f < R.dim; f += kRmsThreads) {
        float s = 0.f;
#pragma unroll
        for (int v = 0; v < kRmsThreads / 64; ++v) s += s_dw[v][f];
        R.partial[(int64_t)blockIdx.x * R.dim + f] = s;
    }
}

template <typename T, int LPR, int ROPE>
__global__ __launch_bounds__(kRmsThreads) void k_rms_bwd(RmsDev R) {
    rms_bwd_rows<T, LPR, ROPE>(R);
}

template <typename T, int LPR, int ROPE>
__global__ __launch_bounds__(kRmsThreads) void k_rms_bwd_many(RmsMany M) {
    rms_bwd_rows<T, LPR, ROPE>(M.it[blockIdx.y]);
}

// dw[f] = sum over the nparts partial rows in a fixed order: the 64 lanes of a wave stride
// the partials, then a fixed butterfly; one wave per feature
__device__ __forceinline__ void rms_dw_sum(const RmsDev& R, int nparts, int dtype) {
    const int lane = threadIdx.x & 63;
    const int f = blockIdx.x * (kRmsThreads / 64) + (threadIdx.x >> 6);
    if (f >= R.dim) return;
    float s[4] = {0.f, 0.f, 0.f, 0.f};  // independent chains: the loads stay in flight
    int p = lane;
    for (; p + 192 < nparts; p += 256)
#pragma unroll
        for (int k = 0; k < 4; ++k) s[k] += R.partial[(int64_t)(p + 64 * k) * R.dim + f];
    for (; p < nparts; p += 64) s[0] += R.partial[(int64_t)p * R.dim + f];
    float t = (s[0] + s[1]) + (s[2] + s[3]);
    for (int off = 32; off > 0; off >>= 1) t += __shfl_xor(t, off);
    if (lane == 0) store_any(R.dw, dtype, f, t);
}

__global__ __launch_bounds__(kRmsThreads) void k_rms_dw(RmsDev R, int nparts) {
    rms_dw_sum(R, nparts, PA_F32);
}

// every tensor's weight gradient, rounded to its weight's dtype
__global__ __launch_bounds__(kRmsThreads) void k_rms_dw_many(RmsMany M, int nparts) {
    const RmsDev& R = M.it[blockIdx.y];
    if (R.partial) rms_dw_sum(R, nparts, R.wdt);
}

// ---------------------------------------------------------------------------------------

static int rms_blocks(const RmsDev& R) {
    const int64_t rpb = (int64_t)(kRmsThreads / R.lpr) * kRmsU;
    const int64_t need = ((int64_t)R.rows + rpb - 1) / rpb;
    return (int)(need < kRmsMaxBlocks ? need : kRmsMaxBlocks);
}

static int rms_setup(const pa_rmsnorm* p, RmsDev& R, bool bwd) {
    if (p->batch < 1 || p->heads < 1 || p->n < 1 || p->dim < 1) return PA_EINVAL;
    const int T = p->x.dtype;
    if (T != PA_F32 && T != PA_F16 && T != PA_BF16) return PA_EINVAL;
    const int es = T == PA_F32 ? 4 : 2, E = 16 / es;
    if (p->dim % E != 0 || p->dim > 64 * E) return PA_EUNSUPPORTED;  // a row is within one wave
    auto view_ok = [&](const pa_view& v) {
        if (!v.ptr || v.dtype != T || v.heads != p->heads) return false;
        return (uintptr_t)v.ptr % 16 == 0 && v.sb % E == 0 && v.sh % E == 0 && v.sn % E == 0;
    };
    if (!view_ok(p->x)) return PA_EINVAL;
    if (!bwd && !view_ok(p->y)) return PA_EINVAL;
    if (bwd && (!view_ok(p->dy) || !view_ok(p->dx))) return PA_EINVAL;
    if (bwd && !p->rstd) return PA_EINVAL;  // the forward writes it only when given
    if (p->weight && p->weight_dtype != PA_F32 && p->weight_dtype != PA_F16 &&
        p->weight_dtype != PA_BF16)
        return PA_EINVAL;
    if (p->angles && (p->rot_dim < 0 || p->rot_dim > p->dim || p->rot_dim % 2 != 0 ||
                      p->angles_stride < 0 ||
                      (p->angles_dtype != PA_F32 && p->angles_dtype != PA_F16 && p->angles_dtype != PA_BF16)))
        return PA_EINVAL;
    int lpr = 1;
    while (lpr * E < p->dim) lpr <<= 1;
    const int64_t rows = (int64_t)p->batch * p->heads * p->n;
    if (rows >= ((int64_t)1 << 31)) return PA_EUNSUPPORTED;
    auto mk = [](const pa_view& v) {
        RView x;
        x.p = static_cast<char*>(v.ptr);
        x.sb = v.sb;
        x.sh = v.sh;
        x.sn = v.sn;
        return x;
    };
    R.batch = p->batch;
    R.heads = p->heads;
    R.n = p->n;
    R.dim = p->dim;
    R.lpr = lpr;
    R.rows = (uint32_t)rows;
    R.hfast = p->heads > 1 && p->n > 1 && p->x.sh < p->x.sn;
    R.fd_n = make_fastdiv((uint32_t)p->n);
    R.fd_h = make_fastdiv((uint32_t)p->heads);
    R.eps = p->eps;
    R.inv_dim = 1.f / (float)p->dim;
    R.x = mk(p->x);
    R.y = mk(p->y);
    R.dy = mk(p->dy);
    R.dx = mk(p->dx);
    R.w = p->weight;
    R.wdt = p->weight_dtype;
    R.rstd = p->rstd;
    R.partial = nullptr;
    R.dw = p->dweight;
    R.ang = (p->angles && p->rot_dim > 0) ? p->angles : nullptr;
    R.adt = p->angles_dtype;
    R.rot_dim = R.ang ? p->rot_dim : 0;
    R.astride = p->angles_stride;
    // the trig table pays where a position's angles serve several rows of a run
    const int rpb = kRmsThreads / lpr, slots = (rpb + p->heads - 2) / p->heads + 1;
    R.trig = R.ang && R.hfast && p->heads >= 4 && kRmsU * slots * R.rot_dim <= kTrigMax ? slots : 0;
    return PA_OK;
}

template <typename T, int ROPE>
static void rms_launch_r(const RmsDev& R, bool bwd, hipStream_t s) {
    const dim3 grid(rms_blocks(R));
#define PA_RMS_CASE(L)                                                                          \
    case L:                                                                                     \
        if (bwd) hipLaunchKernelGGL((k_rms_bwd<T, L, ROPE>), grid, dim3(kRmsThreads), 0, s, R); \
        else hipLaunchKernelGGL((k_rms_fwd<T, L, ROPE>), grid, dim3(kRmsThreads), 0, s, R);     \
        break;
    switch (R.lpr) {
        PA_RMS_CASE(1)
        PA_RMS_CASE(2)
        PA_RMS_CASE(4)
        PA_RMS_CASE(8)
        PA_RMS_CASE(16)
        PA_RMS_CASE(32)
        default: PA_RMS_CASE(64)
    }
#undef PA_RMS_CASE
}

template <typename T>
static void rms_launch(const RmsDev& R, bool bwd, hipStream_t s) {
    if (!R.ang) rms_launch_r<T, kRopeNone>(R, bwd, s);
    else if (R.trig) rms_launch_r<T, kRopeTable>(R, bwd, s);
    else rms_launch_r<T, kRopeRows>(R, bwd, s);
}

int launch_rms_fwd(const pa_rmsnorm* p, hipStream_t s) {
    RmsDev R;
    const int st = rms_setup(p, R, false);
    if (st != PA_OK) return st;
    ProfScope ps("rms_fwd", s);
    if (p->x.dtype == PA_F32) rms_launch<float>(R, false, s);
    else if (p->x.dtype == PA_F16) rms_launch<f16>(R, false, s);
    else rms_launch<bf16>(R, false, s);
    return PA_OK;
}

// the norms of a layer: one dtype, dim and use of angles; the grid's width, or a status < 0
static int rms_many_setup(const pa_rmsnorm* items, int count, bool bwd, RmsMany& M) {
    if (!items || count < 1 || count > PA_RMS_MAX_ITEMS) return PA_EINVAL;
    int blocks = 1;
    for (int k = 0; k < count; ++k) {
        const pa_rmsnorm* p = items + k;
        if (p->x.dtype != items[0].x.dtype || p->dim != items[0].dim) return PA_EINVAL;
        const int st = rms_setup(p, M.it[k], bwd);
        if (st != PA_OK) return st;
        if ((M.it[k].ang != nullptr) != (M.it[0].ang != nullptr)) return PA_EINVAL;
        blocks = std::max(blocks, rms_blocks(M.it[k]));
    }
    return blocks;
}

template <typename T, int ROPE>
static void rms_many_launch_r(const RmsMany& M, dim3 grid, bool bwd, hipStream_t s) {
#define PA_RMS_CASE(L)                                                                               \
    case L:                                                                                          \
        if (bwd) hipLaunchKernelGGL((k_rms_bwd_many<T, L, ROPE>), grid, dim3(kRmsThreads), 0, s, M); \
        else hipLaunchKernelGGL((k_rms_fwd_many<T, L, ROPE>), grid, dim3(kRmsThreads), 0, s, M);     \
        break;
    switch (M.it[0].lpr) {
        PA_RMS_CASE(1)
        PA_RMS_CASE(2)
        PA_RMS_CASE(4)
        PA_RMS_CASE(8)
        PA_RMS_CASE(16)
        PA_RMS_CASE(32)
        default: PA_RMS_CASE(64)
    }
#undef PA_RMS_CASE
}

template <typename T>
static void rms_many_launch_t(const RmsMany& M, int count, dim3 grid, bool bwd, hipStream_t s) {
    int tables = 0;
    for (int k = 0; k < count; ++k) tables += M.it[k].trig != 0;
    if (!M.it[0].ang) rms_many_launch_r<T, kRopeNone>(M, grid, bwd, s);
    else if (tables == count) rms_many_launch_r<T, kRopeTable>(M, grid, bwd, s);
    else if (tables == 0) rms_many_launch_r<T, kRopeRows>(M, grid, bwd, s);
    else rms_many_launch_r<T, kRopeEither>(M, grid, bwd, s);
}

static void rms_many_launch(const RmsMany& M, int dtype, int count, dim3 grid, bool bwd, hipStream_t s) {
    if (dtype == PA_F32) rms_many_launch_t<float>(M, count, grid, bwd, s);
    else if (dtype == PA_F16) rms_many_launch_t<f16>(M, count, grid, bwd, s);
    else rms_many_launch_t<bf16>(M, count, grid, bwd, s);
}

int launch_rms_fwd_many(const pa_rmsnorm* items, int count, hipStream_t s) {
    for (int k = 0; items && k < std::min(count, (int)PA_RMS_MAX_ITEMS); ++k)
        if (items[k].angles) return PA_EUNSUPPORTED;  // rotary: pa_rmsnorm_many
    RmsMany M;
    const int blocks = rms_many_setup(items, count, false, M);
    if (blocks < 0) return blocks;
    ProfScope ps("rms_fwd_many", s);
    rms_many_launch(M, items[0].x.dtype, count, dim3(blocks, count), false, s);
    return PA_OK;
}

size_t rms_many_workspace(const pa_rmsnorm* items, int count) {
    RmsMany M;
    const int blocks = rms_many_setup(items, count, true, M);
    return blocks < 0 ? 0 : (size_t)blocks * count * items[0].dim * sizeof(float);
}

int launch_rms_many(const pa_rmsnorm* items, int count, bool bwd, hipStream_t s) {
    RmsMany M;
    const int blocks = rms_many_setup(items, count, bwd, M);
    if (blocks < 0) return blocks;
    const dim3 grid(blocks, count);
    bool dw = false;
    if (bwd) {
        const size_t each = (size_t)blocks * items[0].dim;
        for (int k = 0; k < count; ++k) {
            if (!items[k].dweight) continue;
            if (!items[0].workspace || items[0].workspace_bytes < each * count * sizeof(float)) return PA_EWORKSPACE;
            M.it[k].partial = static_cast<float*>(items[0].workspace) + k * each;
            if (!items[k].weight) M.it[k].wdt = PA_F32;
            dw = true;
        }
    }
    {
        ProfScope ps(bwd ? "rms_bwd" : "rms_fwd", s);
        rms_many_launch(M, items[0].x.dtype, count, grid, bwd, s);
    }
    if (dw) {
        ProfScope ps("rms_dw", s);
        const int per = kRmsThreads / 64;
        hipLaunchKernelGGL(k_rms_dw_many, dim3((items[0].dim + per - 1) / per, count), dim3(kRmsThreads), 0, s, M,
                           blocks);
    }
    return PA_OK;
}

size_t rms_bwd_workspace(const pa_rmsnorm* p) {
    RmsDev R;
    if (rms_setup(p, R, true) != PA_OK) return 0;
    return (size_t)rms_blocks(R) * p->dim * sizeof(float);
}

int launch_rms_bwd(const pa_rmsnorm* p, hipStream_t s) {
    RmsDev R;
    const int st = rms_setup(p, R, true);
    if (st != PA_OK) return st;
    const int nb = rms_blocks(R);
    if (p->dweight) {
        const size_t need = (size_t)nb * p->dim * sizeof(float);
        if (!p->workspace || p->workspace_bytes < need) return PA_EWORKSPACE;
        R.partial = static_cast<float*>(p->workspace);
    }
    {
        ProfScope ps("rms_bwd", s);
        if (p->x.dtype == PA_F32) rms_launch<float>(R, true, s);
        else if (p->x.dtype == PA_F16) rms_launch<f16>(R, true, s);
        else rms_launch<bf16>(R, true, s);
    }
    if (p->dweight) {
        ProfScope ps("rms_dw", s);
        const dim3 grid((p->dim + kRmsThreads / 64 - 1) / (kRmsThreads / 64));
        hipLaunchKernelGGL(k_rms_dw, grid, dim3(kRmsThreads), 0, s, R, nb);
    }
    return PA_OK;
}

}  // namespace pa
