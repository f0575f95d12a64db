// gemm.hip - the batched-prefill projections on MFMA (gfx950).
//
// Replaces the bf16 -> fp32 weight conversion + cblas_sgemm pairs of the
// reference's batched prefill (gemma3_transformer.c:614-639 Q/K/V, 694-699
// o_proj, 726-751 gate / up / down): C[n][m] = sum_k X[n][k] W[m][k], X the
// fp32 activations of N tokens [N][K], W a bf16 weight matrix [M][K].
//
// Precision.  W is exact in bf16.  X is fp32; it arrives split into two bf16
// planes, x = x_hi + x_lo (x_hi = bf16(x), x_lo = bf16(x - x_hi): 16
// significant bits, relative error <= 2^-17), written by the kernel that
// produces X.  Each product is W.x_hi + W.x_lo on v_mfma_f32_16x16x32_bf16
// with fp32 accumulation: twice the algorithmic MFMA work, within a few
// 2^-17 of the reference's fp32 sgemm.
//
// Tiling.  Three forms of gemm_kernel, picked by g3k_gemm_plan: Pairs (many
// tokens), Quads (many tokens, short rows) and Stream in two widths (few
// tokens); each says what bounds it.  In all of them W and x tiles move from
// global memory straight into LDS with buffer -> LDS loads
// (buffer_load_dwordx4 ... lds, one wave instruction = 1 KiB).  Rows beyond M
// or N read zero (the buffer descriptor's range check), so ragged tiles need
// no masking until the stores.  A row's 16-byte pieces are XOR-swizzled by
// row bits, so a fragment read (16 rows, one piece) spreads over the banks.
// MFMA operands: A = W rows (lane l: row l % 16, k 8 (l / 16) .. + 7), B = X
// rows in the same pattern; the accumulator of lane l holds C rows m = 4 (l /
// 16) + i for token l % 16.
//
// Modes.  PLAIN: up to three weight matrices that share X in one launch (the
// Q, K and V projections), each written as fp32 C [N][ldc].  GEGLU: the gate
// and up matrices together; gelu_tanh(gate) * up (gemma3_transformer.c:741-745)
// is written as the bf16 hi / lo planes that the down projection reads.
#include <hip/hip_runtime.h>

#include "g3k.h"
#include "g3k_device.h"

namespace {

using namespace g3k;

constexpr int BN = 128, BK = 32, NT = 256;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void *lds_ptr;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)bytes, 0x00020000);
}

__device__ __forceinline__ float gelu_tanh(float x) {
    const float inner = 0.7978845608028654f * (x + 0.044715f * (x * x * x));
    return 0.5f * x * (1.0f + tanhf(inner));
}

// bf16 round-to-nearest-even of a finite float, as bits.
__device__ __forceinline__ uint32_t bf16_rne(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}

// Four values of token n at columns m.. as the bf16 hi / lo planes.
__device__ __forceinline__ void store_planes(const g3k_gemm_args &a, int n, int m, float h0, float h1, float h2,
                                             float h3) {
    const float h[4] = {h0, h1, h2, h3};
    uint32_t hi[4], lo[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        hi[i] = bf16_rne(h[i]);
        lo[i] = bf16_rne(h[i] - __uint_as_float(hi[i] << 16));
    }
    const size_t o = (size_t)n * a.ldh + m;
    *reinterpret_cast<uint2 *>(a.h_hi + o) = make_uint2(hi[0] | (hi[1] << 16), hi[2] | (hi[3] << 16));
    *reinterpret_cast<uint2 *>(a.h_lo + o) = make_uint2(lo[0] | (lo[1] << 16), lo[2] | (lo[3] << 16));
}

// One buffer -> LDS fetch of 1 KiB, 16 bytes per lane.  soff (uniform) stays
// below the buffer's size, so the range check covers voff + soff: a lane past
// the end reads zero.
__device__ __forceinline__ void fetch8(__amdgpu_buffer_rsrc_t rs, char *dst, uint32_t voff, uint32_t soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr)dst, 16, voff, soff, 0, 0);
}

// Where matrix m's products of split z go, and their row stride: C, or with
// a.part the columns of the matrices side by side, [split][N][sum of M].
__device__ __forceinline__ float *out_base(const g3k_gemm_args &a, int m, int z, long long &ld) {
    if (!a.part) {
        ld = a.ldc[m];
        return a.C[m] + (size_t)z * a.split_stride;
    }
    int col = 0;
    ld = 0;
    for (int j = 0; j < a.n_mat; j++) {
        if (j < m) col += a.M[j];
        ld += a.M[j];
    }
    return a.part + (size_t)z * a.N * ld + col;
}

// ---------------------------------------------------------------------------
// Many tokens: 256 weight rows (GEGLU: 128 gate rows and the same 128 up
// rows) x 128 tokens per workgroup of 8 waves, one workgroup per CU, K in
// chunks of 64 with two chunks of LDS (2 x 64 KiB).  The eight waves are four
// 128-row x 64-token quarters times two halves of every chunk's k values: a
// wave reads 16 fragments for 64 MFMAs, two waves run per SIMD, and a fetch
// takes whole 128-byte lines (8 rows x 128 B; 16 rows x 64 B halve what an L2
// delivers).  The two k halves meet through LDS at the end, each wave
// finishing half of its pair's tiles.
// Against Quads' tiles (us): down_proj (2560 x 10240) of 8192 / 2048 / 512
// tokens 896 -> 781, 300 -> 193, 79 -> 62; gate and up (2 x 10240 x 2560) of
// 8192 / 2048 / 256 tokens 1509 -> 1422 (1.21 PFLOP/s issued, what a library
// bf16 product of that size reaches here), 447 -> 382, 97 -> 72.  One 64-wide
// stage and two such workgroups per CU: the same at 8192, slower below (gate
// and up of 2048: 407).  The K loop is bound by the matrix cores at the clocks
// they sustain and by the L2 -> LDS stream about equally (down_proj at 8192
// without its fetches: 602; with a quarter of its MFMAs: 645).
template <bool GEGLU>
struct Pairs {
    static constexpr int THREADS = 512, WAVES = 2;
    static __device__ void run(const g3k_gemm_args &a);
};
template <bool GEGLU>
__device__ __forceinline__ void Pairs<GEGLU>::run(const g3k_gemm_args &a) {
    constexpr int MT = 8, NTL = 4, KC = 64;
    constexpr int W_B = 256 * KC * 2, X_B = BN * KC * 2, STAGE_B = W_B + 2 * X_B;
    __shared__ __attribute__((aligned(1024))) char smem[2 * STAGE_B];

    constexpr int BMW = GEGLU ? 128 : 256;               // matrix rows per workgroup
    int bx = blockIdx.x, m_idx = 0;
    if (!GEGLU) {
        while (m_idx + 1 < a.n_mat && bx >= (a.M[m_idx] + BMW - 1) / BMW) {
            bx -= (a.M[m_idx] + BMW - 1) / BMW;
            m_idx++;
        }
    }
    const int M = a.M[m_idx], K = a.K, N = a.N;
    const int m0 = bx * BMW, n0 = blockIdx.y * BN;
    // split z takes chunks [c0, c1) of 64 k values
    const int chunks = (K + KC - 1) / KC;
    const int c0 = (int)((long long)chunks * blockIdx.z / a.ksplit);
    const int c1 = (int)((long long)chunks * (blockIdx.z + 1) / a.ksplit);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave & 1, wn = (wave >> 1) & 1, kw = wave >> 2;
    const int fr = lane & 15, fc = lane >> 4;

    // wave w fetches rows 32 w .. + 31 of the W region and of the two x
    // planes (hi: waves 0..3, lo: 4..7), four instructions each
    const __amdgpu_buffer_rsrc_t rw = rsrc(a.W[GEGLU ? kw : m_idx], (uint32_t)((size_t)M * K * 2));
    const __amdgpu_buffer_rsrc_t rx = rsrc(kw ? a.x_lo : a.x_hi, (uint32_t)((size_t)N * a.ldx * 2));
    const int dr = lane >> 3, dc = ((lane & 7) ^ dr) * 16;
    const uint32_t wvo = (uint32_t)(m0 + (GEGLU ? wave & 3 : wave) * 32 + dr) * (uint32_t)K * 2u + dc;
    const uint32_t xvo = (uint32_t)(n0 + (wave & 3) * 32 + dr) * (uint32_t)a.ldx * 2u + dc;

    f32x4 acc[MT][NTL];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < NTL; nt++) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};

    auto fetch = [&](int s, int c) {
        const uint32_t kb = (uint32_t)c * (KC * 2);
        char *ws = smem + s * STAGE_B + wave * 4096, *xs = ws + W_B;
#pragma unroll
        for (int i = 0; i < 4; i++) fetch8(rw, ws + i * 1024, wvo + (uint32_t)i * (uint32_t)K * 16u, kb);
#pragma unroll
        for (int i = 0; i < 4; i++) fetch8(rx, xs + i * 1024, xvo + (uint32_t)i * (uint32_t)a.ldx * 16u, kb);
    };
    const int f = fr * 128 + (((4 * kw + fc) ^ (fr & 7)) * 16);
    // W region row of the wave's tile mt
    auto wrow = [&](int mt) {
        return GEGLU ? (mt >> 2) * 128 + wm * 64 + (mt & 3) * 16 : wm * 128 + mt * 16;
    };
    fetch(0, c0);
    for (int c = c0; c < c1; c++) {
        const int s = (c - c0) & 1;
        __syncthreads();   // chunk c has landed; the other slot is free
        if (c + 1 < c1) fetch(s ^ 1, c + 1);
        if (c * KC + 32 * kw >= K) continue;   // K ends with half a chunk: nothing for this half
        const char *ws = smem + s * STAGE_B + f, *xs = smem + s * STAGE_B + W_B + wn * (64 * 128) + f;
        bf16x8 h[NTL], l[NTL], w[2];
#pragma unroll
        for (int nt = 0; nt < NTL; nt++) h[nt] = *reinterpret_cast<const bf16x8 *>(xs + nt * 2048);
        w[0] = *reinterpret_cast<const bf16x8 *>(ws + wrow(0) * 128);
#pragma unroll
        for (int nt = 0; nt < NTL; nt++) l[nt] = *reinterpret_cast<const bf16x8 *>(xs + X_B + nt * 2048);
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            // the next W fragment is requested ahead of this one's MFMAs
            if (mt + 1 < MT) w[(mt + 1) & 1] = *reinterpret_cast<const bf16x8 *>(ws + wrow(mt + 1) * 128);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int nt = 0; nt < NTL; nt++)
                acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[mt & 1], h[nt], acc[mt][nt], 0, 0, 0);
#pragma unroll
            for (int nt = 0; nt < NTL; nt++)
                acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[mt & 1], l[nt], acc[mt][nt], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    __syncthreads();

    // lane holds rows m = base + 4 (l / 16) + i, i = 0..3, of token l % 16
    long long ld;
    float *C = GEGLU ? nullptr : out_base(a, m_idx, blockIdx.z, ld);
    f32x4 *red = reinterpret_cast<f32x4 *>(smem);   // 16 KiB per wave: its pair's half of the tiles
    // tile t (0..3) of the half that k half hw finishes
    auto tile = [](int hw, int t) { return GEGLU ? 4 * (t >> 1) + 2 * hw + (t & 1) : 4 * hw + t; };
    auto hand_over = [&](int hw) {
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int nt = 0; nt < NTL; nt++) red[wave * 1024 + (t * NTL + nt) * 64 + lane] = acc[tile(hw, t)][nt];
    };
    if (kw) hand_over(0);
    else hand_over(1);
    __syncthreads();
    auto finish = [&](int hw) {
        const f32x4 *in = red + (wave ^ 4) * 1024 + lane;
#pragma unroll
        for (int t = 0; t < (GEGLU ? 2 : 4); t++) {
            const int mt = tile(hw, t), m = m0 + (GEGLU ? wm * 64 : wm * 128) + mt * 16 + 4 * fc;
#pragma unroll
            for (int nt = 0; nt < NTL; nt++) {
                const int n = n0 + wn * 64 + nt * 16 + fr;
                f32x4 v = in[(t * NTL + nt) * 64];
                v += acc[mt][nt];
                if (GEGLU) {
                    const f32x4 u = acc[tile(hw, t + 2)][nt] + in[((t + 2) * NTL + nt) * 64];
                    if (n < N && m < M)   // M is a multiple of 4 (checked on the host)
                        store_planes(a, n, m, gelu_tanh(v[0]) * u[0], gelu_tanh(v[1]) * u[1], gelu_tanh(v[2]) * u[2],
                                     gelu_tanh(v[3]) * u[3]);
                } else if (n < N && m < M) {
                    *reinterpret_cast<float4 *>(C + (size_t)n * ld + m) = make_float4(v[0], v[1], v[2], v[3]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    if (kw) finish(1);
    else finish(0);
}

// ---------------------------------------------------------------------------
// Short rows (K up to about 2000), or grids of tiles that leave a last round
// nearly empty: 32 MT weight rows x 128 tokens (MT = 4, 8) per workgroup of 4
// waves, a quarter of the tile each, two workgroups per CU, K in stages of 32.
// One's first fetches and last stores (a whole output tile of 64 or 128 KiB)
// run under the other's K loop; with one workgroup per CU, as in Pairs, they
// add to it.  Against Pairs at S = 1 (us): 1024 tokens, 102400 x 96: 149 ->
// 115; 2048 tokens, 12368 x 352: 68 -> 56; 1024, 10240 x 512: 35.0 -> 30.8;
// 2048, 10240 x 2560: 189 -> 202.
// LDS rows are 64 B; within each 16-row group the four 16-byte pieces of row
// r sit at slot 4 r + (c ^ (r / 4 % 4)), so a fragment read (16 rows, one
// piece) touches all 64 banks once.
template <int MT>
struct Quads {
    static constexpr int THREADS = 256, WAVES = 2, ROWS = 32 * MT, TOKENS = BN;
    static constexpr int PART_B = 128 * BK * 2;   // 128 rows of a stage: 8 KiB
    // Rows row0 .. row0 + 127, k0 .. k0 + 31 of a [rows][ld] matrix into LDS:
    // wave w takes the 16-row groups w and w + 4, lane i slot i of a group.
    static __device__ __forceinline__ void fetch(__amdgpu_buffer_rsrc_t rs, char *dst, int row0, int ld, int k0,
                                                 int wave, int lane) {
        const int r = lane >> 2, c = (lane & 3) ^ ((r >> 2) & 3);
#pragma unroll
        for (int g = wave; g < 8; g += 4)
            fetch8(rs, dst + g * 1024, (uint32_t)(row0 + g * 16 + r) * (uint32_t)ld * 2u + c * 16, (uint32_t)k0 * 2u);
    }
    static __device__ __forceinline__ bf16x8 frag(const char *st, int r, int c) {
        return *reinterpret_cast<const bf16x8 *>(st + ((r >> 4) * 64 + (r & 15) * 4 + (c ^ ((r >> 2) & 3))) * 16);
    }
    static __device__ void run(const g3k_gemm_args &a);
};
template <int MT>
__device__ __forceinline__ void Quads<MT>::run(const g3k_gemm_args &a) {
    constexpr int W_B = ROWS * BK * 2, STAGE_B = W_B + 2 * PART_B;
    __shared__ __attribute__((aligned(1024))) char smem[2 * STAGE_B];
    int bx = blockIdx.x, m_idx = 0;
    while (m_idx + 1 < a.n_mat && bx >= (a.M[m_idx] + ROWS - 1) / ROWS) {
        bx -= (a.M[m_idx] + ROWS - 1) / ROWS;
        m_idx++;
    }
    const int M = a.M[m_idx], K = a.K, N = a.N;
    const int m0 = bx * ROWS, n0 = blockIdx.y * BN;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave & 1, wn = wave >> 1;
    const int fr = lane & 15, fc = lane >> 4;
    const __amdgpu_buffer_rsrc_t rw = rsrc(a.W[m_idx], (uint32_t)((size_t)M * K * 2));
    const uint32_t xbytes = (uint32_t)((size_t)N * a.ldx * 2);
    const __amdgpu_buffer_rsrc_t rxh = rsrc(a.x_hi, xbytes), rxl = rsrc(a.x_lo, xbytes);

    f32x4 acc[MT][4];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < 4; nt++) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto fetch_stage = [&](int s, int k0) {
        char *st = smem + s * STAGE_B;
#pragma unroll
        for (int h = 0; h < ROWS / 128; h++) fetch(rw, st + h * PART_B, m0 + 128 * h, K, k0, wave, lane);
        fetch(rxh, st + W_B, n0, a.ldx, k0, wave, lane);
        fetch(rxl, st + W_B + PART_B, n0, a.ldx, k0, wave, lane);
    };
    // split z takes stages [t0, t1) of 32 k values
    const int stages = K / BK;
    const int t0 = (int)((long long)stages * blockIdx.z / a.ksplit);
    const int t1 = (int)((long long)stages * (blockIdx.z + 1) / a.ksplit);
    fetch_stage(0, t0 * BK);
    for (int t = t0; t < t1; t++) {
        const int s = (t - t0) & 1;
        __syncthreads();   // stage t has landed; the other slot is free
        if (t + 1 < t1) fetch_stage(s ^ 1, (t + 1) * BK);
        const char *st = smem + s * STAGE_B;
        bf16x8 h[4], l[4];
#pragma unroll
        for (int nt = 0; nt < 4; nt++) {
            h[nt] = frag(st + W_B, wn * 64 + nt * 16 + fr, fc);
            l[nt] = frag(st + W_B + PART_B, wn * 64 + nt * 16 + fr, fc);
        }
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            const bf16x8 w = frag(st, wm * 16 * MT + mt * 16 + fr, fc);
#pragma unroll
            for (int nt = 0; nt < 4; nt++) {
                acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, h[nt], acc[mt][nt], 0, 0, 0);
                acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, l[nt], acc[mt][nt], 0, 0, 0);
            }
        }
    }
    // lane holds rows m = base + 4 (l / 16) + i, i = 0..3, of token l % 16
    long long ld;
    float *C = out_base(a, m_idx, blockIdx.z, ld);
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < 4; nt++) {
            const int m = m0 + wm * 16 * MT + mt * 16 + 4 * fc, n = n0 + wn * 64 + nt * 16 + fr;
            if (n >= N || m >= M) continue;   // M is a multiple of 4 (checked on the host)
            const f32x4 c = acc[mt][nt];
            *reinterpret_cast<float4 *>(C + (size_t)n * ld + m) = make_float4(c[0], c[1], c[2], c[3]);
        }
}

// ---------------------------------------------------------------------------
// Few tokens: the weight stream.
//
// With N <= 128 tokens (a short message, a ragged tail) the projection is one
// pass over W at the HBM rate; 128 x 128 tiles leave most CUs idle (down_proj:
// 20 workgroups) and walk K in 0.6 us steps.  Here a workgroup of NWV waves
// covers 16 MT NWV weight rows x 16 NTL tokens, every wave its own 16 MT rows
// and all the tokens, and K is split until the grid fills the chip.  K moves
// in chunks of 64: one DMA instruction takes 8 rows x 128 B (a whole line of
// each row: 16 rows x 64 B, the MFMA operand's own shape, read W at 2.3-4.0
// TB/s against 5.0-5.5), and the next chunks are in flight in two LDS rings, DW
// slots of W and DX of x, whose barrier waits only for the oldest.  Where two
// chunks of 96 or 128 tokens fill the LDS, x (from the L2) keeps two slots and
// W (from memory) takes the rest as a third: gate and up of 77 tokens, 2 x
// 10240 x 2560: 32.4 -> 30.0 us.  (One workgroup of 128 rows x 96 or 128
// tokens with these rings instead of 64 rows x 48 or 64, for the other
// products: down_proj of 100 tokens 21.1 -> 26.0 us, twice the splits.)  A row's eight 16-byte pieces sit at
// c ^ (row % 8), so a fragment read (16 rows, one piece) spreads over the
// banks.  Rows past M or N read zero; rows of a last half chunk past K hold
// other rows' values and are not multiplied.
// Every split writes fp32 partial products; the consumer or
// split_reduce_kernel adds them in split order.
template <int MT, int NTL, int DW, int DX, int NWV, int OCC>
struct Stream {
    static constexpr int THREADS = NWV * 64, WAVES = OCC, ROWS = NWV * MT * 16, TOKENS = NTL * 16;
    static __device__ void run(const g3k_gemm_args &a);
};
template <int MT, int NTL, int DW, int DX, int NWV, int OCC>
__device__ __forceinline__ void Stream<MT, NTL, DW, DX, NWV, OCC>::run(const g3k_gemm_args &a) {
    constexpr int BM = NWV * MT * 16, KC = 64;
    constexpr int W_B = BM * KC * 2, X_B = NTL * 16 * KC * 2;   // X_B: one plane
    constexpr int NWI = MT * 2;             // W fetches of a wave per chunk (8 rows each)
    constexpr int NXI = NTL * 4 / NWV;      // its x_hi / x_lo fetches
    static_assert(NTL * 4 % NWV == 0, "every wave issues the same number of fetches (counted waits)");
    static_assert(DX >= 2 && (DW == DX || DW == DX + 1), "a deeper W ring would drain at x's wait");
    __shared__ __attribute__((aligned(1024))) char smem[DW * W_B + DX * 2 * X_B];

    int bx = blockIdx.x, m_idx = 0;
    while (m_idx + 1 < a.n_mat && bx >= (a.M[m_idx] + BM - 1) / BM) {
        bx -= (a.M[m_idx] + BM - 1) / BM;
        m_idx++;
    }
    const int M = a.M[m_idx], K = a.K, N = a.N;
    const int m0 = bx * BM, n0 = blockIdx.y * (NTL * 16);
    // split z takes chunks [c0, c1) of 64 k values
    const int chunks = (K + KC - 1) / KC;
    const int c0 = (int)((long long)chunks * blockIdx.z / a.ksplit);
    const int c1 = (int)((long long)chunks * (blockIdx.z + 1) / a.ksplit);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int fr = lane & 15, fc = lane >> 4;

    const __amdgpu_buffer_rsrc_t rw = rsrc(a.W[m_idx], (uint32_t)((size_t)M * K * 2));
    const uint32_t xbytes = (uint32_t)((size_t)N * a.ldx * 2);
    const __amdgpu_buffer_rsrc_t rxh = rsrc(a.x_hi, xbytes), rxl = rsrc(a.x_lo, xbytes);
    // this lane's 16 bytes of a fetch: row lane / 8, piece (lane % 8) ^ row
    const int dr = lane >> 3, dc = ((lane & 7) ^ dr) * 16;
    const uint32_t wbase = (uint32_t)(m0 + wave * MT * 16 + dr) * (uint32_t)K * 2u + dc;
    const uint32_t xbase = (uint32_t)(n0 + dr) * (uint32_t)a.ldx * 2u + dc;

    f32x4 acc[MT][NTL];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < NTL; nt++) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};

    // W and x of chunk c (clamped to the split's last: the counted waits want
    // every round to issue the same number) into slot s of their rings
    auto fetch_w = [&](int s, int c) {
        const uint32_t kb = (uint32_t)(c < c1 ? c : c1 - 1) * (KC * 2);
        char *ws = smem + s * W_B + wave * (MT * 2048);
#pragma unroll
        for (int i = 0; i < NWI; i++) fetch8(rw, ws + i * 1024, wbase + (uint32_t)i * (uint32_t)K * 16u, kb);
    };
    auto fetch_x = [&](int s, int c) {
        const uint32_t kb = (uint32_t)(c < c1 ? c : c1 - 1) * (KC * 2);
        char *xs = smem + DW * W_B + s * (2 * X_B);
#pragma unroll
        for (int j = 0; j < NXI; j++) {
            const int g = wave + NWV * j, r8 = g % (2 * NTL);   // 8-row group r8 of plane g / (2 NTL)
            fetch8(g < 2 * NTL ? rxh : rxl, xs + g * 1024, xbase + (uint32_t)r8 * (uint32_t)a.ldx * 16u, kb);
        }
    };
    // The rings' waits count fetches in issue order, so no round may move
    // into another: a scheduling fence after each.  The round of chunk c
    // fetches x of chunk c + DX - 1, then W of chunk c + DW - 1.  With DW >
    // DX the wait for chunk c leaves the W fetched after its x in flight, so
    // there a round's x comes before its W: a fence between them too.
    auto x_first = [] {
        if (DW > DX) G3K_ORDER_FENCE();
    };
#pragma unroll
    for (int d = 1 - DW; d < 0; d++) {
        if (d + DX - 1 >= 0) fetch_x(d + DX - 1, c0 + d + DX - 1);
        x_first();
        fetch_w(d + DW - 1, c0 + d + DW - 1);
        G3K_ORDER_FENCE();
    }
    const int f0 = fr * 128 + ((fc ^ (fr & 7)) * 16), f1 = fr * 128 + (((4 + fc) ^ (fr & 7)) * 16);
    int sw = 0, sx = 0;
    for (int c = c0; c < c1; c++) {
        // chunk c has landed (the DX - 2 rounds after its x, and the W fetched
        // after it, may be in flight) and every wave is done with chunk c - 1,
        // whose slots are filled next
        G3K_WAIT_BARRIER((DX - 2) * (NWI + NXI) + (DW > DX ? NWI : 0));
        fetch_x(sx == 0 ? DX - 1 : sx - 1, c + DX - 1);
        x_first();
        fetch_w(sw == 0 ? DW - 1 : sw - 1, c + DW - 1);
        G3K_ORDER_FENCE();
        const char *ws = smem + sw * W_B + wave * (MT * 2048), *xs = smem + DW * W_B + sx * (2 * X_B);
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {
            if (kk == 1 && c * KC + 32 >= K) break;   // uniform: K ends with half a chunk
            const int f = kk ? f1 : f0;
            bf16x8 w[MT];
#pragma unroll
            for (int mt = 0; mt < MT; mt++) w[mt] = *reinterpret_cast<const bf16x8 *>(ws + mt * 2048 + f);
#pragma unroll
            for (int nt = 0; nt < NTL; nt++) {
                const bf16x8 xh = *reinterpret_cast<const bf16x8 *>(xs + nt * 2048 + f);
                const bf16x8 xl = *reinterpret_cast<const bf16x8 *>(xs + X_B + nt * 2048 + f);
#pragma unroll
                for (int mt = 0; mt < MT; mt++)
                    acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[mt], xh, acc[mt][nt], 0, 0, 0);
#pragma unroll
                for (int mt = 0; mt < MT; mt++)
                    acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[mt], xl, acc[mt][nt], 0, 0, 0);
            }
        }
        sw = sw + 1 == DW ? 0 : sw + 1;
        sx = sx + 1 == DX ? 0 : sx + 1;
    }
    // the clamped fetches past the end still write the ring
    G3K_WAIT_VMEM();

    // lane holds rows m = base + 4 (l / 16) + i, i = 0..3, of token l % 16
    long long ld;
    float *C = out_base(a, m_idx, blockIdx.z, ld);
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < NTL; nt++) {
            const int m = m0 + wave * MT * 16 + mt * 16 + 4 * fc, n = n0 + nt * 16 + fr;
            if (n >= N || m >= M) continue;   // M is a multiple of 4 (checked on the host)
            const f32x4 c = acc[mt][nt];
            *reinterpret_cast<float4 *>(C + (size_t)n * ld + m) = make_float4(c[0], c[1], c[2], c[3]);
        }
}

// One launch of form F (Stream, Pairs, Quads).
template <class F>
__global__ __launch_bounds__(F::THREADS, F::WAVES) void gemm_kernel(g3k_gemm_args a) {
    F::run(a);
}

// Adds the partial products a.part [ksplit][N][sum of M] in split order into
// C (plain) or, for GEGLU, into the hi / lo planes of gelu_tanh(gate) * up.
// One thread per four columns of one token (GEGLU: of gate and up).
template <bool GEGLU>
__global__ __launch_bounds__(NT) void split_reduce_kernel(g3k_gemm_args a) {
    int ld = 0;
    for (int j = 0; j < a.n_mat; j++) ld += a.M[j];
    const int n = blockIdx.x, m = 4 * (blockIdx.y * NT + threadIdx.x);
    if (m >= (GEGLU ? a.M[0] : ld)) return;
    const size_t stride = (size_t)a.N * ld;
    auto sum = [&](int col) {
        const float4 *p = reinterpret_cast<const float4 *>(a.part + (size_t)n * ld + col);
        float4 t = *p;
#pragma unroll 8
        for (int s = 1; s < a.ksplit; s++) {
            const float4 v = *reinterpret_cast<const float4 *>(a.part + s * stride + (size_t)n * ld + col);
            t = make_float4(t.x + v.x, t.y + v.y, t.z + v.z, t.w + v.w);
        }
        return t;
    };
    if (GEGLU) {
        const float4 g = sum(m), u = sum(a.M[0] + m);
        store_planes(a, n, m, gelu_tanh(g.x) * u.x, gelu_tanh(g.y) * u.y, gelu_tanh(g.z) * u.z, gelu_tanh(g.w) * u.w);
        return;
    }
    int j = 0, col = m;
    while (j + 1 < a.n_mat && col >= a.M[j]) col -= a.M[j++];
    *reinterpret_cast<float4 *>(a.C[j] + (size_t)n * a.ldc[j] + col) = sum(m);
}

// Workgroups of `rows` weight rows that cover the launch's matrices.
int row_tiles(const g3k_gemm_args *a, int rows) {
    int tiles = 0;
    for (int m = 0; m < a->n_mat; m++) tiles += (a->M[m] + rows - 1) / rows;
    return tiles;
}

int launch_reduce(const g3k_gemm_args *a, hipStream_t st) {
    const bool geglu = a->mode == G3K_MV_GEGLU;
    int cols = a->M[0];
    for (int m = 1; m < a->n_mat && !geglu; m++) cols += a->M[m];
    const dim3 grid(a->N, (cols / 4 + NT - 1) / NT);
    if (geglu)
        hipLaunchKernelGGL((split_reduce_kernel<true>), grid, dim3(NT), 0, st, *a);
    else
        hipLaunchKernelGGL((split_reduce_kernel<false>), grid, dim3(NT), 0, st, *a);
    return (int)hipGetLastError();
}

template <class F>
int launch(const g3k_gemm_args *a, int tiles, int blocks, hipStream_t st) {
    hipLaunchKernelGGL((gemm_kernel<F>), dim3(tiles, blocks, a->ksplit), dim3(F::THREADS), 0, st, *a);
    return (int)hipGetLastError();
}

template <class F>
int launch_stream(const g3k_gemm_args *a, hipStream_t st) {
    return launch<F>(a, row_tiles(a, F::ROWS), (a->N + F::TOKENS - 1) / F::TOKENS, st);
}

// Tokens per workgroup of the 64-row stream: 48 where that covers N in as many
// blocks as 64 does.
int narrow_tokens(int N) {
    return N <= 16 ? 16 : N <= 32 ? 32 : (N + 47) / 48 == (N + 63) / 64 ? 48 : 64;
}

int launch_form(const g3k_gemm_args *a, hipStream_t st) {
    const int nb = (a->N + BN - 1) / BN;
    switch (a->kind) {
        case G3K_GEMM_WIDE:
            if (a->N <= 32) return launch_stream<Stream<2, 2, 3, 3, 8, 1>>(a, st);
            if (a->N <= 64) return launch_stream<Stream<2, 4, 3, 3, 8, 1>>(a, st);
            if (a->N <= 96) return launch_stream<Stream<2, 6, 3, 2, 8, 1>>(a, st);
            return launch_stream<Stream<2, 8, 3, 2, 8, 1>>(a, st);
        case G3K_GEMM_NARROW:
            if (a->N <= 16) return launch_stream<Stream<1, 1, 5, 5, 4, 2>>(a, st);
            if (a->N <= 32) return launch_stream<Stream<1, 2, 3, 3, 4, 2>>(a, st);
            if (narrow_tokens(a->N) == 48) return launch_stream<Stream<1, 3, 3, 3, 4, 2>>(a, st);
            return launch_stream<Stream<1, 4, 2, 2, 4, 3>>(a, st);
        case G3K_GEMM_QUAD128:
            return launch_stream<Quads<4>>(a, st);
        case G3K_GEMM_QUAD256:
            return launch_stream<Quads<8>>(a, st);
        default:
            if (a->mode == G3K_MV_GEGLU) return launch<Pairs<true>>(a, (a->M[0] + 127) / 128, nb, st);
            return launch<Pairs<false>>(a, row_tiles(a, 256), nb, st);
    }
}

}  // namespace

namespace {

// A form's time, in us at 256 CUs, as fitted to 5500 measured products (N 1 to
// 4097, M 4 to 262208, K 32 to 10240; each form within 5 to 12% rms):
//   2.3 + rounds (round + chunk[o - 1] chunks) + w_read W MB per token block
//   + out C MB (+ 3.3 + 0.32 S C MB for split sums that a second launch adds)
// A round is per_cu workgroups on every CU; o, how many share a CU in it.
// tokens: the most a row of the table holds for (Stream's token classes).
struct FormTime {
    int kind, rows, tokens, per_cu;
    double round, chunk[3], w_read, out;
};
constexpr FormTime FORMS[] = {
    {G3K_GEMM_NARROW, 64, 16, 2, 0.68, {0.18, 0.50, 0}, 0.044, 0.178},
    {G3K_GEMM_NARROW, 64, 32, 2, 0.54, {0.30, 0.55, 0}, 0.049, 0.084},
    {G3K_GEMM_NARROW, 64, 48, 2, 0.62, {0.30, 0.55, 0}, 0.051, 0.150},
    {G3K_GEMM_NARROW, 64, 64, 3, 0.59, {0.42, 0.49, 0.73}, 0.075, 0.108},
    {G3K_GEMM_WIDE, 256, 64, 1, 0.85, {0.67, 0, 0}, 0.111, 0.214},
    {G3K_GEMM_WIDE, 256, 96, 1, 1.17, {0.99, 0, 0}, 0.078, 0.227},
    {G3K_GEMM_WIDE, 256, 128, 1, 1.92, {1.34, 0, 0}, 0.059, 0.197},
    {G3K_GEMM_TILE, 256, 128, 1, 2.19, {1.23, 0, 0}, 0.040, 0.180},
    {G3K_GEMM_QUAD128, 128, 128, 2, 0.54, {1.05, 1.21, 0}, 0.077, 0.168},
    {G3K_GEMM_QUAD256, 256, 128, 2, 1.34, {1.74, 2.70, 0}, 0.035, 0.166},
};

double form_time(const FormTime &f, int N, int K, int n_mat, const int *M, int S, int cus) {
    long long tiles = 0, sum = 0;
    for (int m = 0; m < n_mat; m++) {
        tiles += (M[m] + f.rows - 1) / f.rows;
        sum += M[m];
    }
    const long long blocks = (N + f.tokens - 1) / f.tokens, wgs = tiles * blocks * S, slots = (long long)cus * f.per_cu;
    // the quads walk stages of 32, the others chunks of 64
    const int all = (K + 63) / 64;
    const bool quad = f.kind == G3K_GEMM_QUAD128 || f.kind == G3K_GEMM_QUAD256;
    const double chunks = quad ? K / 64.0 / S : (double)((all + S - 1) / S);
    const long long full = wgs / slots, rest = wgs % slots;
    double t = 2.27 + (double)full * (f.round + f.chunk[f.per_cu - 1] * chunks);
    if (rest) t += f.round + f.chunk[(rest + cus - 1) / cus - 1] * chunks;
    const double out_mb = 4e-6 * N * (double)sum;
    t += f.w_read * 2e-6 * (double)sum * K * (double)blocks + f.out * out_mb;
    return S > 1 ? t + 3.27 + 0.32 * S * out_mb : t;
}

}  // namespace

// The kernel and its k splits for N tokens.
// - GEGLU: up to 128 tokens the 256-row stream, split until there is a
//   workgroup per CU; beyond, the tiles unsplit.
// - Partial products that the consumer adds (the residual step, which reads
//   them anyway): the 64-row stream up to 128 tokens or 12 GFLOP issued, split
//   to two workgroups per CU (it is ahead there, 384 tokens of 2560 x 2560 take
//   20 us against 27, level with the tiles from 13 to 20 and behind from 27
//   GFLOP: 256 tokens of 2560 x 10240 51 against 47, 1024 of 2560 x 2560 40
//   against 39); beyond, the tiles, whose split z adds its part to
//   the time of a round of n_cu workgroups (1.75 us per 64-wide chunk and 5 us
//   around the K loop, measured with every CU busy) and its partial products
//   (moved at about 8 MB per us); the S with the least total is taken.
// - Otherwise the form and S of the least time above.  The candidates: the
//   64-row stream in the range just given, unless a second token block would
//   read W from memory again (more than two workgroups of one block per CU);
//   the 256-row stream for 49 to 128 tokens over many rows; the tiles, split
//   beyond 128 tokens; the quads.  One rule for all of them left 710 of the
//   5500 products 10 to 88% over the earlier 128 x 128 tiles (a batch's logits
//   in one call, 128 tokens, 262208 x 2560: 772 us for 423; 1024 tokens,
//   102400 x 96: 145 for 112); with the times 25 are, by at most 21%.
//   A split has at least two chunks, and its partial products at most 256 MB.
extern "C" void g3k_gemm_plan(int N, int K, int n_mat, const int *M, int geglu, int consumer_adds, int n_cu, int *kind,
                              int *ksplit) {
    long long sum = 0, tiles64 = 0, tiles256 = 0;
    for (int m = 0; m < n_mat; m++) {
        sum += M[m];
        tiles64 += (M[m] + 63) / 64;
        tiles256 += (M[m] + 255) / 256;
    }
    const int chunks = (K + 63) / 64, most = chunks > 1 ? chunks / 2 : 1;
    const int cus = n_cu > 0 ? n_cu : 256;
    const bool stream = N <= 128 || (N <= 4096 && 4.0 * N * (double)sum * K <= 12e9);
    const long long tiles = tiles256 * ((N + BN - 1) / BN);
    const int per = narrow_tokens(N);
    const long long wgs64 = tiles64 * ((N + per - 1) / per);
    auto bounded = [&](long long S) { return (int)(S < 1 ? 1 : S > most ? most : S); };
    auto room = [&](int S) { return S == 1 || 4.0 * S * N * (double)sum <= 256e6; };
    *kind = G3K_GEMM_TILE;
    *ksplit = 1;
    if (geglu) {
        if (N > 128) return;
        *kind = G3K_GEMM_WIDE;
        *ksplit = bounded(cus / tiles256);
        return;
    }
    if (consumer_adds && stream) {
        *kind = G3K_GEMM_NARROW;
        *ksplit = bounded(2LL * cus / wgs64);
        return;
    }
    double best = 0.0;
    if (consumer_adds) {
        for (int s = 1; s <= 16 && s <= most && room(s); s++) {
            double t = (double)((tiles * s + cus - 1) / cus) * (1.75 * ((chunks + s - 1) / s) + 5.0);
            if (s > 1) t += (double)s * N * (double)sum * 8.0 / 8e6;
            if (s == 1 || t < best) {
                best = t;
                *ksplit = s;
            }
        }
        return;
    }
    for (const FormTime &f : FORMS) {
        int tried = 0;
        auto consider = [&](int S) {
            if (S == tried || !room(S)) return;
            tried = S;
            double t = form_time(f, N, K, n_mat, M, S, cus);
            // whole 128-byte lines of W: the 64-row stream's fit is over its
            // measured times there (5.2 M outputs at K = 512: 20 against 17)
            if (f.kind == G3K_GEMM_NARROW && K % 64 == 0 && K >= 256) t *= 0.85;
            if (best > 0.0 && t >= best) return;
            best = t;
            *kind = f.kind;
            *ksplit = S;
        };
        switch (f.kind) {
            case G3K_GEMM_NARROW:
                if (!stream || f.tokens != per || (N > per && tiles64 > 2 * cus)) break;
                for (int j = 0; j <= 3; j++) consider(bounded((long long)j * cus / wgs64));
                break;
            case G3K_GEMM_WIDE:
                if (N <= 48 || N > f.tokens || N <= f.tokens - (f.tokens == 64 ? 16 : 32) || tiles256 <= cus / 4) break;
                consider(1);
                consider(bounded(cus / tiles256));
                break;
            case G3K_GEMM_TILE:
                for (int s = 1; s <= 16 && s <= most && (s == 1 || N > 128); s++) consider(s);
                break;
            default:
                consider(1);
        }
    }
}

extern "C" int g3k_gemm(const g3k_gemm_args *a, void *stream) {
    const bool geglu = a->mode == G3K_MV_GEGLU;
    const int S = a->ksplit;
    if (a->N < 1 || a->K < BK || a->K % BK || a->ldx < a->K || a->ldx % 8 || !a->x_hi || !a->x_lo)
        return (int)hipErrorInvalidValue;
    if (a->n_mat < 1 || a->n_mat > G3K_MATVEC_MAX || (geglu && a->n_mat != 2) || (a->mode != 0 && !geglu))
        return (int)hipErrorInvalidValue;
    if (a->kind < G3K_GEMM_TILE || a->kind > G3K_GEMM_QUAD256) return (int)hipErrorInvalidValue;
    // at least one 64-wide chunk per split; the grid's y and z limits
    const bool stream_w = a->kind == G3K_GEMM_WIDE || a->kind == G3K_GEMM_NARROW;
    if (S < 1 || S > (a->K + 63) / 64 || S > 65535 || a->N > (stream_w ? 16 : BN) * 65535)
        return (int)hipErrorInvalidValue;
    // GEGLU is applied to whole sums: through part, or by an unsplit tile kernel
    if (geglu && (stream_w ? !a->part : (S != 1 || a->part || a->kind != G3K_GEMM_TILE))) return (int)hipErrorInvalidValue;
    // 32-bit buffer offsets, including the rows of a last partial tile
    if ((size_t)(a->N + BN) * a->ldx * 2 >= (1ull << 32)) return (int)hipErrorInvalidValue;
    for (int m = 0; m < a->n_mat; m++) {
        if (a->M[m] < 4 || a->M[m] % 4 || !a->W[m] || (size_t)(a->M[m] + 256) * a->K * 2 >= (1ull << 32))
            return (int)hipErrorInvalidValue;
        if (geglu) continue;
        if (!a->C[m] || a->ldc[m] < a->M[m] || a->ldc[m] % 4) return (int)hipErrorInvalidValue;
        if (S > 1 && !a->part && a->split_stride < (long long)a->N * a->ldc[m]) return (int)hipErrorInvalidValue;
    }
    if (geglu && (a->M[0] != a->M[1] || !a->h_hi || !a->h_lo || a->ldh < a->M[0] || a->ldh % 4))
        return (int)hipErrorInvalidValue;
    hipStream_t st = (hipStream_t)stream;
    const int rc = launch_form(a, st);
    return rc || !a->part ? rc : launch_reduce(a, st);
}
