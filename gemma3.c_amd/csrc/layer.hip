// layer.hip - the small kernels between the GEMVs of one token's forward pass
// (gemma3_transformer_forward, gemma3_transformer.c:396-512): the embedding
// row, the hidden-size RMSNorms with their residual adds.
//
// Each works on one hidden vector (a few thousand floats), so each is one
// workgroup: latency, not bandwidth, is what they cost, and folding the
// norms and adds that sit between two GEMVs into one launch is what matters.
//   embed:     x = bf16(E[token]) * sqrt(hidden)          (:415-422)
//   norm:      y = rmsnorm(x, w)                           (:444-446, 508)
//   residual:  t = rmsnorm(t, w_post)  (if w_post)         (:463-466, 490-493)
//              x = x + t                                   (:469, 496)
//              y = rmsnorm(x, w_next)  (if y; a copy of x if w_next is NULL)
// rmsnorm is gemma3_rmsnorm_bf16 (gemma3_kernels.c:289-304): mean of squares
// + eps, 1 / sqrtf, then x * r * (1 + bf16(w)); the sum of squares is a tree
// here instead of the reference's sequential loop.
#include <hip/hip_runtime.h>

#include "g3k.h"
#include "g3k_device.h"

namespace {

using namespace g3k;

constexpr int NT = 1024;
constexpr int NW = NT / 64;
constexpr int PER = 8;   // values per thread: hidden <= NT * PER

// Sum over the workgroup; every thread gets the total.
__device__ __forceinline__ float block_sum(float v, float *red) {
    v = wave_sum(v);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    __syncthreads();   // red may still be read by an earlier call
    if (lane == 0) red[wave] = v;
    __syncthreads();
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < NW; w++) s += red[w];
    return s;
}

// r = 1 / sqrtf(mean(v^2) + eps) over the n values held PER per thread.
__device__ __forceinline__ float rms_scale(const float (&v)[PER], int n, float eps, float *red) {
    float ss = 0.f;
#pragma unroll
    for (int u = 0; u < PER; u++) ss += v[u] * v[u];
    ss = block_sum(ss, red);
    return 1.0f / sqrtf(ss / (float)n + eps);
}

__global__ __launch_bounds__(NT) void embed_kernel(g3k_layer_args a) {
    const int n = a.n;
    const float scale = sqrtf((float)n);
    const uint16_t *row = a.embed + (size_t)a.token * n;
    for (int i = threadIdx.x; i < n; i += NT) a.x[i] = bf16f(row[i]) * scale;
}

// The gains (1 + w) of a norm, loaded up front so that their latency overlaps
// the activations' loads instead of following a reduction.
__device__ __forceinline__ void load_gain(float (&g)[PER], const uint16_t *w, int n) {
#pragma unroll
    for (int u = 0; u < PER; u++) {
        const int i = threadIdx.x + NT * u;
        g[u] = (w && i < n) ? 1.0f + bf16f(w[i]) : 0.f;
    }
}

__global__ __launch_bounds__(NT) void norm_kernel(g3k_layer_args a) {
    __shared__ float red[NW];
    const int n = a.n;
    float v[PER], g[PER];
    load_gain(g, a.w_next, n);
#pragma unroll
    for (int u = 0; u < PER; u++) {
        const int i = threadIdx.x + NT * u;
        v[u] = i < n ? a.x[i] : 0.f;
    }
    const float r = rms_scale(v, n, a.eps, red);
#pragma unroll
    for (int u = 0; u < PER; u++) {
        const int i = threadIdx.x + NT * u;
        if (i < n) a.y[i] = v[u] * r * g[u];
    }
}

__global__ __launch_bounds__(NT) void residual_kernel(g3k_layer_args a) {
    __shared__ float red[NW];
    const int n = a.n;
    float t[PER], x[PER], gp[PER], gn[PER];
    load_gain(gp, a.w_post, n);
    load_gain(gn, a.y ? a.w_next : nullptr, n);
#pragma unroll
    for (int u = 0; u < PER; u++) {
        const int i = threadIdx.x + NT * u;
        t[u] = i < n ? a.t[i] : 0.f;
        x[u] = i < n ? a.x[i] : 0.f;
    }
    if (a.w_post) {
        const float r = rms_scale(t, n, a.eps, red);
#pragma unroll
        for (int u = 0; u < PER; u++) t[u] = t[u] * r * gp[u];   // gp is 0 past n
    }
#pragma unroll
    for (int u = 0; u < PER; u++) {
        const int i = threadIdx.x + NT * u;
        x[u] = x[u] + t[u];
        if (i < n) a.x[i] = x[u];
    }
    if (!a.y) return;   // uniform
    if (a.w_next) {
        const float r = rms_scale(x, n, a.eps, red);
#pragma unroll
        for (int u = 0; u < PER; u++) {
            const int i = threadIdx.x + NT * u;
            if (i < n) a.y[i] = x[u] * r * gn[u];
        }
    } else {
#pragma unroll
        for (int u = 0; u < PER; u++) {
            const int i = threadIdx.x + NT * u;
            if (i < n) a.y[i] = x[u];
        }
    }
}

}  // namespace

extern "C" int g3k_layer_step(const g3k_layer_args *a, void *stream) {
    if (a->n < 1 || a->n > G3K_LAYER_MAX_HIDDEN) return (int)hipErrorInvalidValue;
    hipStream_t st = (hipStream_t)stream;
    switch (a->op) {
        case G3K_OP_EMBED:
            if (!a->embed || !a->x || a->token < 0) return (int)hipErrorInvalidValue;
            hipLaunchKernelGGL(embed_kernel, dim3(1), dim3(NT), 0, st, *a);
            break;
        case G3K_OP_NORM:
            if (!a->x || !a->y || !a->w_next) return (int)hipErrorInvalidValue;
            hipLaunchKernelGGL(norm_kernel, dim3(1), dim3(NT), 0, st, *a);
            break;
        case G3K_OP_RESIDUAL:
            if (!a->x || !a->t) return (int)hipErrorInvalidValue;
            hipLaunchKernelGGL(residual_kernel, dim3(1), dim3(NT), 0, st, *a);
            break;
        default:
            return (int)hipErrorInvalidValue;
    }
    return (int)hipGetLastError();
}

// ------------------------------------------------------------ batched rows
// One workgroup of 256 threads per token row (gemma3_transformer.c:585-592,
// 596-602, 702-724, 753-765: the reference's per-token loops of the batched
// prefill).  Thread i holds the PER 4-element groups i + 256 u, PER fixed per
// row length, so every load of a row (its k splits, residual and gains) is a
// 16-byte one requested before the first use.  A short batch is a handful of
// rows whose cost is that one round trip (77 rows of 2560 with 6 splits: 23
// -> 7 us against 32 masked 4-byte loads per thread and split), a long one
// moves its rows at the HBM rate.  Rows that are not a multiple of 4 values
// or not 16-byte aligned take 4-byte accesses in the same order.

namespace {

constexpr int RNT = 256;
constexpr int RNW = RNT / 64;

__device__ __forceinline__ float rblock_sum(float v, float *red) {
    v = wave_sum(v);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    __syncthreads();
    if (lane == 0) red[wave] = v;
    __syncthreads();
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < RNW; w++) s += red[w];
    return s;
}

__device__ __forceinline__ uint32_t rne16(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}

// Group g (values 4 g .. 4 g + 3) of a row of n values; past the end 0.
template <bool VEC>
__device__ __forceinline__ float4 load4(const float *p, int g, int n) {
    const int i = 4 * g;
    if (VEC) {
        const float4 v = reinterpret_cast<const float4 *>(p)[i < n ? g : 0];
        return i < n ? v : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    return make_float4(i < n ? p[i] : 0.f, i + 1 < n ? p[i + 1] : 0.f, i + 2 < n ? p[i + 2] : 0.f,
                       i + 3 < n ? p[i + 3] : 0.f);
}

template <bool VEC>
__device__ __forceinline__ void store4(float *p, int g, int n, float4 v) {
    const int i = 4 * g;
    if (VEC) {
        if (i < n) reinterpret_cast<float4 *>(p)[g] = v;
        return;
    }
    if (i < n) p[i] = v.x;
    if (i + 1 < n) p[i + 1] = v.y;
    if (i + 2 < n) p[i + 2] = v.z;
    if (i + 3 < n) p[i + 3] = v.w;
}

// Four bf16 values; al8: the array is 8-byte aligned (uniform).
template <bool VEC>
__device__ __forceinline__ float4 load_bf4(const uint16_t *p, int g, int n, bool al8) {
    const int i = 4 * g;
    if (VEC && al8) {
        const uint2 w = reinterpret_cast<const uint2 *>(p)[i < n ? g : 0];
        const float4 v = make_float4(bf16f(w.x & 0xffff), bf16f(w.x >> 16), bf16f(w.y & 0xffff), bf16f(w.y >> 16));
        return i < n ? v : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    return make_float4(i < n ? bf16f(p[i]) : 0.f, i + 1 < n ? bf16f(p[i + 1]) : 0.f, i + 2 < n ? bf16f(p[i + 2]) : 0.f,
                       i + 3 < n ? bf16f(p[i + 3]) : 0.f);
}

__device__ __forceinline__ bool aligned8(const void *p) { return ((uintptr_t)p & 7) == 0; }

// y as bf16 hi / lo planes
template <bool VEC>
__device__ __forceinline__ void store_split(const g3k_rows_args &a, int row, int g, float4 y) {
    const float v[4] = {y.x, y.y, y.z, y.w};
    uint32_t hi[4], lo[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        hi[j] = rne16(v[j]);
        lo[j] = rne16(v[j] - __uint_as_float(hi[j] << 16));
    }
    uint16_t *yh = a.y_hi + (size_t)row * a.ldy + 4 * g, *yl = a.y_lo + (size_t)row * a.ldy + 4 * g;
    if (VEC) {
        if (4 * g >= a.n) return;
        *reinterpret_cast<uint2 *>(yh) = make_uint2(hi[0] | hi[1] << 16, hi[2] | hi[3] << 16);
        *reinterpret_cast<uint2 *>(yl) = make_uint2(lo[0] | lo[1] << 16, lo[2] | lo[3] << 16);
        return;
    }
#pragma unroll
    for (int j = 0; j < 4; j++)
        if (4 * g + j < a.n) {
            yh[j] = (uint16_t)hi[j];
            yl[j] = (uint16_t)lo[j];
        }
}

__device__ __forceinline__ float4 scale4(float4 v, float r, float4 w) {
    return make_float4(v.x * r * (1.0f + w.x), v.y * r * (1.0f + w.y), v.z * r * (1.0f + w.z), v.w * r * (1.0f + w.w));
}
__device__ __forceinline__ float4 add4(float4 a, float4 b) {
    return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
}

// 1 / sqrtf(mean(v^2) + eps) of the row held PER groups per thread (0 past its end)
template <int PER>
__device__ __forceinline__ float row_scale(const float4 (&v)[PER], int n, float eps, float *red) {
    float ss = 0.f;
#pragma unroll
    for (int u = 0; u < PER; u++) ss += v[u].x * v[u].x + v[u].y * v[u].y + v[u].z * v[u].z + v[u].w * v[u].w;
    return 1.0f / sqrtf(rblock_sum(ss, red) / (float)n + eps);
}

template <int PER, bool VEC>
__global__ __launch_bounds__(RNT) void rows_kernel(g3k_rows_args a) {
    __shared__ float red[RNW];
    const int row = blockIdx.x, n = a.n, tid = threadIdx.x;
    if (a.op == G3K_ROWS_SPLIT) {   // elementwise: any row length, over gridDim.y workgroups
        const float *t = a.t + (size_t)row * a.ldt;
        const int step = RNT * gridDim.y;
        for (int g = tid + RNT * blockIdx.y; 4 * g < n; g += step) store_split<VEC>(a, row, g, load4<VEC>(t, g, n));
        return;
    }
    float *x = a.x + (size_t)row * n;
    float4 v[PER], gn[PER];
    const bool next = a.w_next && a.y_hi;
    if (next) {
#pragma unroll
        for (int u = 0; u < PER; u++) gn[u] = load_bf4<VEC>(a.w_next, tid + RNT * u, n, aligned8(a.w_next));
    }
    if (a.op == G3K_ROWS_EMBED) {
        const float scale = sqrtf((float)n);
        const uint16_t *e = a.embed + (size_t)a.tokens[row] * n;
#pragma unroll
        for (int u = 0; u < PER; u++) {
            const float4 b = load_bf4<VEC>(e, tid + RNT * u, n, aligned8(e));
            v[u] = make_float4(b.x * scale, b.y * scale, b.z * scale, b.w * scale);
            store4<VEC>(x, tid + RNT * u, n, v[u]);
        }
    } else {
        const float *t = a.t + (size_t)row * a.ldt;
        float4 tv[PER], gp[PER];
#pragma unroll
        for (int u = 0; u < PER; u++) {
            tv[u] = load4<VEC>(t, tid + RNT * u, n);
            v[u] = load4<VEC>(x, tid + RNT * u, n);
        }
        if (a.w_post) {
#pragma unroll
            for (int u = 0; u < PER; u++) gp[u] = load_bf4<VEC>(a.w_post, tid + RNT * u, n, aligned8(a.w_post));
        }
        // the k splits of the producing GEMM, added in order, four at a time
        for (int s = 1; s < a.nsplit; s += 4) {
            float4 p[4][PER];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float *ts = t + (size_t)min(s + j, a.nsplit - 1) * a.split_stride;
#pragma unroll
                for (int u = 0; u < PER; u++) p[j][u] = load4<VEC>(ts, tid + RNT * u, n);
            }
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (s + j < a.nsplit) {
#pragma unroll
                    for (int u = 0; u < PER; u++) tv[u] = add4(tv[u], p[j][u]);
                }
        }
        if (a.w_post) {
            const float r = row_scale<PER>(tv, n, a.eps, red);
#pragma unroll
            for (int u = 0; u < PER; u++) tv[u] = scale4(tv[u], r, gp[u]);   // 0 past n
        }
#pragma unroll
        for (int u = 0; u < PER; u++) {
            v[u] = add4(v[u], tv[u]);
            store4<VEC>(x, tid + RNT * u, n, v[u]);
        }
        if (!a.y_hi) return;   // uniform
    }
    if (next) {
        const float r = row_scale<PER>(v, n, a.eps, red);
#pragma unroll
        for (int u = 0; u < PER; u++) v[u] = scale4(v[u], r, gn[u]);
    }
#pragma unroll
    for (int u = 0; u < PER; u++) store_split<VEC>(a, row, tid + RNT * u, v[u]);
}

template <int PER>
void launch_rows(const g3k_rows_args *a, bool vec, hipStream_t st) {
    // the split has no row sum: a workgroup per 1024 values, so that a few long
    // rows are one round trip of the whole chip instead of a loop per row (100
    // rows of 10240 into a projection: the call 30.5 -> 27.9 us)
    const int parts = a->op == G3K_ROWS_SPLIT ? min((int)((a->n + 4LL * RNT - 1) / (4 * RNT)), 64) : 1;
    const dim3 grid(a->rows, parts);
    if (vec)
        hipLaunchKernelGGL((rows_kernel<PER, true>), grid, dim3(RNT), 0, st, *a);
    else
        hipLaunchKernelGGL((rows_kernel<PER, false>), grid, dim3(RNT), 0, st, *a);
}

bool aligned(const void *p, size_t b) { return ((uintptr_t)p & (b - 1)) == 0; }

}  // namespace

extern "C" int g3k_rows(const g3k_rows_args *a, void *stream) {
    if (a->rows < 1 || a->n < 1 || (a->op != G3K_ROWS_SPLIT && a->n > G3K_LAYER_MAX_HIDDEN))
        return (int)hipErrorInvalidValue;
    const bool split_out = a->y_hi && a->y_lo && a->ldy >= a->n;
    switch (a->op) {
        case G3K_ROWS_EMBED:
            if (!a->tokens || !a->embed || !a->x || !split_out) return (int)hipErrorInvalidValue;
            break;
        case G3K_ROWS_RESIDUAL:
            if (!a->x || !a->t || a->ldt < a->n || ((a->y_hi || a->y_lo) && !split_out) || a->nsplit < 1 ||
                (a->nsplit > 1 && a->split_stride < (long long)a->rows * a->ldt))
                return (int)hipErrorInvalidValue;
            break;
        case G3K_ROWS_SPLIT:
            if (!a->t || a->ldt < a->n || !split_out) return (int)hipErrorInvalidValue;
            break;
        default:
            return (int)hipErrorInvalidValue;
    }
    const bool has_x = a->op != G3K_ROWS_SPLIT, has_t = a->op != G3K_ROWS_EMBED;
    const bool vec = a->n % 4 == 0 && (!has_x || aligned(a->x, 16)) &&
                     (!has_t || (aligned(a->t, 16) && a->ldt % 4 == 0 && (a->nsplit < 2 || a->split_stride % 4 == 0))) &&
                     (!a->y_hi || (aligned(a->y_hi, 8) && aligned(a->y_lo, 8) && a->ldy % 4 == 0));
    hipStream_t st = (hipStream_t)stream;
    const int per = a->op == G3K_ROWS_SPLIT ? 1 : (a->n + 4 * RNT - 1) / (4 * RNT);
    switch (per) {
        case 1: launch_rows<1>(a, vec, st); break;
        case 2: launch_rows<2>(a, vec, st); break;
        case 3: launch_rows<3>(a, vec, st); break;
        case 4: launch_rows<4>(a, vec, st); break;
        default: launch_rows<8>(a, vec, st); break;
    }
    return (int)hipGetLastError();
}
