// Row projections  Y[R][N] = X[R][K] . W[N][K]^T  with F16 weights and F32
// activations: the Q/K/V/output projections either side of the attention
// path (reference: wri_op_matmul at src/core/session.c:446-457 and :499-506,
// inner loops src/core/kernels.c:124-137; weights are W[out][in] with `in`
// contiguous, src/core/internal.h:113-118, and F16 tensors are widened to F32
// before the multiply, src/core/loader.c:164-190).
//
// Decode sends 1..16 rows through a projection, so the work is reading W once:
// HBM-bound, algorithmic bytes per launch = 2 * N * K.  The multiply-adds run
// on v_mfma_f32_16x16x32_f16 to keep them off the vector ALUs, as in the decode
// kernel, and F32 accuracy is kept the same way: each row is scaled by a power
// of two into [1, 2) (by its largest magnitude), split into two half-precision
// terms x = hi + lo * 2^-11, and the two terms take two COLUMNS of the same MFMA
// (column c = hi of row c, column c + 8 = lo of row c, eight rows per MFMA).
// The columns are combined and the scale undone at the end; sums are F32.
//
// Layouts on the device (both private to the library):
//
//   W   [N/16][K/32][64][8] halves: tile (nt, kt) is the MFMA A operand of
//       outputs 16nt..16nt+15 and inputs 32kt..32kt+31 in lane order (lane =
//       16g + m holds W[16nt + m][32kt + 8g .. +8]), one contiguous KiB per
//       operand load; a wave streams the K/32 consecutive KiBs of its outputs.
//   X   fragments [ceil(R/8)][K/32][64][8] halves, the matching B operands
//       (lane 16g + c: column c, inputs 32kt + 8g .. +8), and one F32 scale
//       per row, written by proj_prep_kernel, read by every wave (L2 / L1 hits).
//
// Kernels, by row count of a launch:
//   1 row        proj_row1_kernel: the fragment step inside the product;
//   2 .. 16      proj_prep_kernel, then proj_gemm_split_kernel where four waves share
//                a tile's inputs and they are few or the weight small, proj_rows_kernel
//                (a wave owns one or two 16-output tiles for one or two row groups;
//                HBM-bound) elsewhere;
//   17 .. 4096   proj_prep_kernel (proj_prep_group_kernel from 257 rows), then a
//                GEMM: proj_gemm_lds_kernel (operands staged through LDS,
//                MFMA-bound) where its tiles fill the chip,
//                proj_gemm_split_kernel below that.
// N must be a multiple of 16 and K a multiple of 32.
#pragma once

#include <type_traits>

#include "common.hip.h"

namespace wr {

constexpr int kProjThreads = 256;
constexpr int kProjMaxRows = 4096;                // rows per launch (512 row groups)
constexpr int kProjKBatch = 8;                    // k-steps (KiBs of W) a wave keeps in flight per buffer

// Row-major F16 W[N][K] -> tile order.  One thread per 16-byte unit.
__global__ __launch_bounds__(256) void proj_pack_weights_kernel(const uint16_t* __restrict__ w,
                                                                u32x4* __restrict__ tiles,
                                                                uint32_t N, uint32_t K)
{
    const size_t unit = (size_t)blockIdx.x * blockDim.x + threadIdx.x;     // destination unit
    const size_t total = (size_t)N * K / 8;
    if (unit >= total) return;
    const uint32_t lane = (uint32_t)(unit & 63);
    const size_t tile = unit >> 6;
    const uint32_t kt = (uint32_t)(tile % (K / 32));
    const uint32_t nt = (uint32_t)(tile / (K / 32));
    const uint32_t m = lane & 15, g = lane >> 4;
    const u32x4* src = reinterpret_cast<const u32x4*>(w + ((size_t)(nt * 16 + m) * K + kt * 32 + g * 8));
    tiles[unit] = *src;
}

// Rows of the weight as F32 rows, times `scale` where it is not one (an embedding table, which a tied head's weight is):
// a workgroup to a row, a chunk of eight inputs to a thread.  The tokens travel as arguments.  Against rows made on the
// host and sent up (a copy, and the wait for it): a session's step 593 -> 579 us, 2047 rows of 1024 8.38 -> 8.06 ms.
constexpr uint32_t kEmbedTokens = 960;            // of a launch: 4 KiB of arguments

struct ProjEmbedArgs {
    const half8* w;          // tile order
    float* x;                // [rows][ldx]
    uint32_t ldx, K;
    float scale;
    uint32_t tokens[kEmbedTokens];
};

__global__ __launch_bounds__(128) void proj_embed_kernel(const ProjEmbedArgs a)
{
    const uint32_t token = a.tokens[blockIdx.x], ktiles = a.K / 32;
    const half8* w = a.w + (size_t)(token / 16) * ktiles * 64 + token % 16;
    float* x = a.x + (size_t)blockIdx.x * a.ldx;
    for (uint32_t q = threadIdx.x; q < a.K / 8; q += 128) {
        const half8 h = w[(q / 4) * 64 + (q % 4) * 16];
        f32x4 lo, hi;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            lo[j] = (float)h[j] * a.scale;
            hi[j] = (float)h[4 + j] * a.scale;
        }
        *reinterpret_cast<f32x4*>(x + q * 8) = lo;
        *reinterpret_cast<f32x4*>(x + q * 8 + 4) = hi;
    }
}

// X rows -> B-operand fragments and per-row scales, one workgroup per row
// (rows past R, which pad the last group of eight, get zero fragments).
//
// The row is first brought to its final F32 values v[k] by one of three
// sources, so that a normalisation or activation that only feeds a projection
// never has to be written out:
//   kProjSrcPlain    v = x
//   kProjSrcRmsNorm  v = x * (1 / sqrt(mean x^2 + eps)) * w     (RMSNorm,
//                    src/core/kernels.c:1276-1316, same expressions and the
//                    same reduction tree as rmsnorm_rows_kernel)
//   kProjSrcSwiglu   v = silu(g) * u, g = x[k], u = x[K + k]   (kernels.c:963-967)
//   kProjSrcGeglu    v = gelu_tanh(g) * u, same operands      (kernels.c:969-976)
// Then scales[row] = 2^e with 2^e <= max|v| < 2^(e+1) (1 for a row of zeros),
// v is divided by it (exact), so its largest magnitude lies in [1, 2), and
// split into
//   hi = binary16(v), flushed to zero below the normal range, and
//   lo = binary16((v - hi) * 2^11),
// i.e. v = hi + lo * 2^-11 to about 2^-22 |v| (2^-25 of the row's largest value
// for elements so small that hi is flushed).  Keeping lo scaled up keeps both
// terms in the normal binary16 range, so the result does not depend on how the
// matrix cores treat subnormal inputs.
constexpr float kProjLoScale = 2048.0f;
constexpr int kProjSrcPlain = 0, kProjSrcRmsNorm = 1, kProjSrcSwiglu = 2, kProjSrcGeglu = 3;

struct ProjPrepArgs {
    const float* x;          // [R][ldx]
    const float* norm_w;     // kProjSrcRmsNorm: [K]
    half8* frag;             // [groups][K/32][64]
    float* scales;           // [R]
    uint32_t ldx, R, K;
    float eps;
};

// (The barriers in these two wait for LDS traffic only: __syncthreads() would
// also wait for every global load in flight, and the one-row product has its
// weights on the way while it reduces.)
// s4 must not be written again before the workgroup's next barrier (the two
// reductions of a row use the two halves of an array of eight): one barrier
// each, not two.
__device__ __forceinline__ float block_sum_256(float v, float* s4)
{
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += wave_xor_f32(v, off);
    if ((threadIdx.x & 63) == 0) s4[threadIdx.x >> 6] = v;
    lds_barrier();
    return (s4[0] + s4[1]) + (s4[2] + s4[3]);
}

__device__ __forceinline__ float block_max_256(float v, float* s4)
{
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v = fmaxf(v, wave_xor_f32(v, off));
    if ((threadIdx.x & 63) == 0) s4[threadIdx.x >> 6] = v;
    lds_barrier();
    return fmaxf(fmaxf(s4[0], s4[1]), fmaxf(s4[2], s4[3]));
}

// Sum of squares of a row by a 256-thread workgroup.  Thread t takes the
// chunks of eight values t, t + 256, ... in order; the partial sums go through
// a wave tree and the four waves are added pairwise.  Every kernel that
// normalises a row uses this order, so a norm computed inside the fragment
// kernel has the bits of rmsnorm_rows_kernel.
__device__ __forceinline__ float row_sumsq_256(const float* __restrict__ xr, uint32_t K, float* s4)
{
    float ss = 0.f;
    for (uint32_t k0 = threadIdx.x * 8; k0 < K; k0 += 2048) {
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const float v = (k0 + j < K) ? xr[k0 + j] : 0.f;
            ss = fmaf(v, v, ss);          // explicit, so every copy of this sum rounds alike
        }
    }
    return block_sum_256(ss, s4);
}

// the two gated activations: SiLU(g) * u and the tanh form of GELU(g) * u
template <int SRC>
__device__ __forceinline__ float proj_gated(float g, float u)
{
    if constexpr (SRC == kProjSrcGeglu) {
        const float x3 = g * g * g;
        const float z = 0.7978845608f * (g + 0.044715f * x3);
        const float th = 2.0f / (1.0f + expf(-2.0f * z)) - 1.0f;
        return 0.5f * g * (1.0f + th) * u;
    } else {
        return silu_mul(g, u);
    }
}

template <int SRC>
__device__ __forceinline__ float proj_src_value(const ProjPrepArgs& a, const float* xr, uint32_t k,
                                                float inv_rms)
{
    if constexpr (SRC == kProjSrcRmsNorm) {
        return xr[k] * inv_rms * a.norm_w[k];
    } else if constexpr (SRC == kProjSrcSwiglu || SRC == kProjSrcGeglu) {
        return proj_gated<SRC>(xr[k], xr[a.K + k]);
    } else {
        return xr[k];
    }
}

__device__ __forceinline__ void proj_write_chunk(half8* frow, uint32_t q, uint32_t c,
                                                 const float (&v)[8], float inv)
{
    half8 hi, lo;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const float s = v[j] * inv;
        _Float16 h = (_Float16)s;
        if (fabsf((float)h) < 6.103515625e-05f) h = (_Float16)0.0f;      // 2^-14
        hi[j] = h;
        lo[j] = (_Float16)((s - (float)h) * kProjLoScale);
    }
    const uint32_t kt = q >> 2, g = q & 3;
    frow[(size_t)kt * 64 + 16 * g + c] = hi;
    frow[(size_t)kt * 64 + 16 * g + c + 8] = lo;
}

// CH > 0: K <= 2048 * CH and the row's values are held in registers between
// the passes (one read of the row: a single-row call is pure latency, and each
// pass over global memory is a round trip).  CH = 0: any K, the passes re-read
// (and re-compute) the row.
template <int SRC, int CH>
__global__ __launch_bounds__(256) void proj_prep_kernel(const ProjPrepArgs a)
{
    __shared__ float s4[8];
    const uint32_t row = blockIdx.x, t = threadIdx.x;
    const uint32_t ktiles = a.K / 32, nchunks = a.K / 8;
    const uint32_t grp = row / 8, c = row % 8;
    half8* frow = a.frag + (size_t)grp * ktiles * 64;
    if (row >= a.R) {                                     // padding row of the last group
        half8 z;
#pragma unroll
        for (int j = 0; j < 8; j++) z[j] = (_Float16)0.0f;
        for (uint32_t q = t; q < nchunks; q += 256) {
            const uint32_t kt = q >> 2, g = q & 3;
            frow[(size_t)kt * 64 + 16 * g + c] = z;
            frow[(size_t)kt * 64 + 16 * g + c + 8] = z;
        }
        return;
    }
    const float* xr = a.x + (size_t)row * a.ldx;

    if constexpr (CH > 0) {
        float v[CH][8];
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < CH; i++) {
            const uint32_t q = t + 256 * i;
#pragma unroll
            for (int j = 0; j < 8; j++) v[i][j] = (q < nchunks) ? xr[q * 8 + j] : 0.f;
            if constexpr (SRC == kProjSrcRmsNorm) {
#pragma unroll
                for (int j = 0; j < 8; j++) ss = fmaf(v[i][j], v[i][j], ss);
            }
        }
        float mx = 0.f;
        if constexpr (SRC == kProjSrcRmsNorm) {
            const float inv_rms = 1.0f / sqrtf(block_sum_256(ss, s4) / (float)a.K + a.eps);
#pragma unroll
            for (int i = 0; i < CH; i++) {
                const uint32_t q = t + 256 * i;
#pragma unroll
                for (int j = 0; j < 8; j++)
                    v[i][j] = (q < nchunks) ? v[i][j] * inv_rms * a.norm_w[q * 8 + j] : 0.f;
            }
        } else if constexpr (SRC == kProjSrcSwiglu || SRC == kProjSrcGeglu) {
#pragma unroll
            for (int i = 0; i < CH; i++) {
                const uint32_t q = t + 256 * i;
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const float u = (q < nchunks) ? xr[a.K + q * 8 + j] : 0.f;
                    v[i][j] = proj_gated<SRC>(v[i][j], u);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < CH; i++)
#pragma unroll
            for (int j = 0; j < 8; j++) mx = fmaxf(mx, fabsf(v[i][j]));
        mx = block_max_256(mx, s4 + 4);
        uint32_t ex = (__float_as_uint(mx) >> 23) & 0xFFu;
        if (ex == 0 || ex == 0xFF) ex = 127;              // zeros, subnormals, inf / NaN rows: no scaling
        if (ex > 253) ex = 253;                           // keeps the inverse 2^-e a normal number
        if (t == 0) a.scales[row] = __uint_as_float(ex << 23);
        const float inv = __uint_as_float((254u - ex) << 23);
#pragma unroll
        for (int i = 0; i < CH; i++) {
            const uint32_t q = t + 256 * i;
            if (q < nchunks) proj_write_chunk(frow, q, c, v[i], inv);
        }
    } else {
        float inv_rms = 1.0f;
        if constexpr (SRC == kProjSrcRmsNorm)
            inv_rms = 1.0f / sqrtf(row_sumsq_256(xr, a.K, s4) / (float)a.K + a.eps);
        float mx = 0.f;
        for (uint32_t k = t; k < a.K; k += 256) mx = fmaxf(mx, fabsf(proj_src_value<SRC>(a, xr, k, inv_rms)));
        mx = block_max_256(mx, s4 + 4);
        uint32_t ex = (__float_as_uint(mx) >> 23) & 0xFFu;
        if (ex == 0 || ex == 0xFF) ex = 127;
        if (ex > 253) ex = 253;
        if (t == 0) a.scales[row] = __uint_as_float(ex << 23);
        const float inv = __uint_as_float((254u - ex) << 23);
        for (uint32_t q = t; q < nchunks; q += 256) {     // 8 consecutive inputs per thread
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = proj_src_value<SRC>(a, xr, q * 8 + j, inv_rms);
            proj_write_chunk(frow, q, c, v, inv);
        }
    }
}

// The fragment kernel for many rows: one workgroup per row GROUP of eight.
// Thread t serves row t % 8 of the group and the chunks of eight inputs t / 8,
// t / 8 + 32, ...: a wave reads 256 contiguous bytes of each of its eight rows
// per step and writes the hi and lo terms of eight chunks as whole 128-byte
// lines (the eight rows' 16-byte units of one chunk are neighbours in the
// fragment), where the one-row kernel's writes touch 16 bytes of a line each.
// Same sources, expressions and scaling as proj_prep_kernel; the row sums are
// formed in a different order (each thread over its own chunks, then the 32
// threads of the row), so a normalised row agrees with the one-row kernel's to
// rounding, not bit for bit: only launches of many rows come here.
//
// CH > 0: K <= 256 * CH and the row group's values stay in registers between
// the passes, asked for once and all together (with the norm's weights: 2047 rows of
// 1024 8.7 -> 6.8 us; plain rows of 3072, 50 MB, 11.7 us, are at the memory's rate);
// CH = 0: any K, the passes re-read and re-compute.
__device__ __forceinline__ float group_rows_sum(float v, float (*s)[8], int lane, int wave, int c)
{
    v += wave_xor_f32(v, 8);
    v += wave_xor_f32(v, 16);
    v += wave_xor_f32(v, 32);
    if (lane < 8) s[wave][lane] = v;
    __syncthreads();
    const float t = (s[0][c] + s[1][c]) + (s[2][c] + s[3][c]);
    __syncthreads();
    return t;
}

__device__ __forceinline__ float group_rows_max(float v, float (*s)[8], int lane, int wave, int c)
{
    v = fmaxf(v, wave_xor_f32(v, 8));
    v = fmaxf(v, wave_xor_f32(v, 16));
    v = fmaxf(v, wave_xor_f32(v, 32));
    if (lane < 8) s[wave][lane] = v;
    __syncthreads();
    const float t = fmaxf(fmaxf(s[0][c], s[1][c]), fmaxf(s[2][c], s[3][c]));
    __syncthreads();
    return t;
}

// the eight values of chunk q of a row, from the row's source
template <int SRC>
__device__ __forceinline__ void proj_src_chunk(const ProjPrepArgs& a, const float* xr, uint32_t q,
                                               float inv_rms, float (&v)[8])
{
    const f32x4 lo = *reinterpret_cast<const f32x4*>(xr + q * 8), hi = *reinterpret_cast<const f32x4*>(xr + q * 8 + 4);
#pragma unroll
    for (int j = 0; j < 4; j++) {
        v[j] = lo[j];
        v[4 + j] = hi[j];
    }
    if constexpr (SRC == kProjSrcRmsNorm) {
        const f32x4 wl = *reinterpret_cast<const f32x4*>(a.norm_w + q * 8),
                    wh = *reinterpret_cast<const f32x4*>(a.norm_w + q * 8 + 4);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            v[j] = v[j] * inv_rms * wl[j];
            v[4 + j] = v[4 + j] * inv_rms * wh[j];
        }
    } else if constexpr (SRC == kProjSrcSwiglu || SRC == kProjSrcGeglu) {
        const f32x4 ul = *reinterpret_cast<const f32x4*>(xr + a.K + q * 8),
                    uh = *reinterpret_cast<const f32x4*>(xr + a.K + q * 8 + 4);
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = proj_gated<SRC>(v[j], j < 4 ? ul[j] : uh[j - 4]);
    }
}

template <int SRC, int CH>
__global__ __launch_bounds__(256) void proj_prep_group_kernel(const ProjPrepArgs a)
{
    __shared__ float s48[4][8];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int c = t & 7;
    const uint32_t col = t >> 3;                                  // 0..31
    const uint32_t grp = blockIdx.x, row = grp * 8 + c;
    const uint32_t ktiles = a.K / 32, nchunks = a.K / 8;
    half8* frow = a.frag + (size_t)grp * ktiles * 64;
    const bool live = row < a.R;                                  // rows past R pad the last group with zeros
    const float* xr = a.x + (size_t)(live ? row : a.R - 1) * a.ldx;

    // rows need 16-byte alignment for the vector loads: ldx and K are multiples
    // of four floats (the host checks), the base comes from the allocator.
    // The row's values (and, where there is room, the norm's weights or the gates'
    // partners) are asked for all at once and stay (a chunk past the end re-reads the
    // last one; dropped below).
    constexpr bool NORM = SRC == kProjSrcRmsNorm, TWO = SRC != kProjSrcPlain;
    constexpr bool EARLY = TWO && CH <= 8;
    constexpr int HELD = CH > 0 ? CH : 1;
    f32x4 held[HELD][2], with[EARLY ? HELD : 1][2];
    auto partner = [&](uint32_t q, f32x4 (&e)[2]) {
        const float* from = (NORM ? a.norm_w : xr + a.K) + q * 8;
        e[0] = *reinterpret_cast<const f32x4*>(from);
        e[1] = *reinterpret_cast<const f32x4*>(from + 4);
    };
    if constexpr (CH > 0) {
#pragma unroll
        for (int i = 0; i < CH; i++) {
            const uint32_t q = min(col + 32 * i, nchunks - 1);
            held[i][0] = *reinterpret_cast<const f32x4*>(xr + q * 8);
            held[i][1] = *reinterpret_cast<const f32x4*>(xr + q * 8 + 4);
        }
        if constexpr (EARLY) {
#pragma unroll
            for (int i = 0; i < CH; i++) partner(min(col + 32 * i, nchunks - 1), with[i]);
        }
    }
    float inv_rms = 1.0f;
    if constexpr (NORM) {
        float ss = 0.f;
        if constexpr (CH > 0) {
#pragma unroll
            for (int i = 0; i < CH; i++)
                if (col + 32 * i < nchunks) {
#pragma unroll
                    for (int j = 0; j < 8; j++) ss = fmaf(held[i][j / 4][j % 4], held[i][j / 4][j % 4], ss);
                }
        } else {
            for (uint32_t q = col; q < nchunks; q += 32) {
                const f32x4 lo = *reinterpret_cast<const f32x4*>(xr + q * 8), hi = *reinterpret_cast<const f32x4*>(xr + q * 8 + 4);
#pragma unroll
                for (int j = 0; j < 4; j++) ss = fmaf(lo[j], lo[j], ss);
#pragma unroll
                for (int j = 0; j < 4; j++) ss = fmaf(hi[j], hi[j], ss);
            }
        }
        inv_rms = 1.0f / sqrtf(group_rows_sum(ss, s48, lane, wave, c) / (float)a.K + a.eps);
    }

    float mx = 0.f;
    if constexpr (CH > 0) {
#pragma unroll
        for (int i = 0; i < CH; i++) {
            const uint32_t q = col + 32 * i;
            f32x4 e[2];
            if constexpr (EARLY) {
                e[0] = with[i][0];
                e[1] = with[i][1];
            } else if constexpr (TWO) {
                partner(min(q, nchunks - 1), e);
            }
#pragma unroll
            for (int j = 0; j < 8; j++) {
                float v = held[i][j / 4][j % 4];
                if constexpr (NORM)
                    v = v * inv_rms * e[j / 4][j % 4];
                else if constexpr (TWO)
                    v = proj_gated<SRC>(v, e[j / 4][j % 4]);
                held[i][j / 4][j % 4] = v;
                if (q < nchunks) mx = fmaxf(mx, fabsf(v));
            }
        }
    } else {
        for (uint32_t q = col; q < nchunks; q += 32) {
            float v[8];
            proj_src_chunk<SRC>(a, xr, q, inv_rms, v);
#pragma unroll
            for (int j = 0; j < 8; j++) mx = fmaxf(mx, fabsf(v[j]));
        }
    }
    mx = group_rows_max(mx, s48, lane, wave, c);
    uint32_t ex = (__float_as_uint(mx) >> 23) & 0xFFu;
    if (ex == 0 || ex == 0xFF) ex = 127;              // zeros, subnormals, inf / NaN rows: no scaling
    if (ex > 253) ex = 253;                           // keeps the inverse 2^-e a normal number
    if (col == 0 && live) a.scales[row] = __uint_as_float(ex << 23);
    const float inv = __uint_as_float((254u - ex) << 23);

    if constexpr (CH > 0) {
#pragma unroll
        for (int i = 0; i < CH; i++) {
            const uint32_t q = col + 32 * i;
            if (q < nchunks) {
                float v[8];
#pragma unroll
                for (int j = 0; j < 8; j++) v[j] = live ? held[i][j / 4][j % 4] : 0.f;
                proj_write_chunk(frow, q, c, v, inv);
            }
        }
    } else {
        for (uint32_t q = col; q < nchunks; q += 32) {
            float v[8];
            proj_src_chunk<SRC>(a, xr, q, inv_rms, v);
            if (!live) {
#pragma unroll
                for (int j = 0; j < 8; j++) v[j] = 0.f;
            }
            proj_write_chunk(frow, q, c, v, inv);
        }
    }
}

// One 64-byte line, and ProjPrepArgs behind it within the next: the first thing a launch
// of a decode step does is fetch these through the scalar cache.  With 72 bytes, which
// put the second structure across a line's end, a step of a 28-layer model took 925 to
// 1000 us from run to run instead of 885 to 895.
struct ProjArgs {
    const half8* w;          // tile order
    const half8* xfrag;      // [groups][K/32][64]
    const float* scales;     // [R]
    const float* bias_rows;  // optional [R][ldy] added to the result (residual), or nullptr
    float* y;                // [R][ldy]
    uint32_t N, K, R, ldy;
    uint8_t ksplit;          // waves of a workgroup that share one run of outputs: 1, 2 or 4
    uint8_t cols;            // proj_gemm_lds_kernel: XCDs that share out the outputs (xcd_tile)
    uint8_t gate;            // GATED kernels: kProjSrcSwiglu or kProjSrcGeglu
};
static_assert(sizeof(ProjArgs) == 64 && sizeof(ProjPrepArgs) <= 64, "a line each");

// Writes one accumulator tile.  Layout: lane 16g + c holds outputs 16nt + 4g .. +3
// of column c; column c (< 8) is the hi term of row c of the group, column c + 8
// its lo term.  The two are combined, the row's scale undone, the optional
// residual added.  Tiles past N and rows past R are dropped.
__device__ __forceinline__ f32x4 proj_join_terms(f32x4 v)
{
#pragma unroll
    for (int i = 0; i < 4; i++) {
        // the lo column of row c is eight lanes on in the same row of sixteen: a
        // rotation by eight inside the row (DPP row_ror:8), no trip through LDS
        const float other = __int_as_float(
            __builtin_amdgcn_update_dpp(0, __float_as_int(v[i]), 0x128, 0xF, 0xF, false));
        v[i] += other * (1.0f / kProjLoScale);      // meaningful in the hi columns only
    }
    return v;
}

template <int ROWS = 8>
__device__ __forceinline__ void proj_store_tile(const ProjArgs& a, f32x4 v, uint32_t nt, uint32_t group,
                                                int lane, const float* scale = nullptr,
                                                const f32x4* residual = nullptr)
{
    const int c = lane & 15, g = lane >> 4;
    v = proj_join_terms(v);
    const uint32_t row = group * ROWS + (c & 7);
    if (c < ROWS && row < a.R && nt < a.N / 16) {
        const float sc = scale ? *scale : a.scales[row];
        const size_t o = (size_t)row * a.ldy + nt * 16 + g * 4;
        f32x4 r;
#pragma unroll
        for (int i = 0; i < 4; i++) r[i] = v[i] * sc;
        if (a.bias_rows) {
            // (residual: the same values, read earlier by the caller)
            const f32x4 b = residual ? *residual : *reinterpret_cast<const f32x4*>(a.bias_rows + o);
#pragma unroll
            for (int i = 0; i < 4; i++) r[i] += b[i];
        }
        *reinterpret_cast<f32x4*>(a.y + o) = r;
    }
}

// GATED kernels take a weight whose first half of outputs are gates, the second the
// values they gate: tile p and tile p + N / 32 are worked on by the same wave, and
// what is stored is act(gate) * value, [R][N / 2].  The next product then reads half
// the bytes and has no activation to work out (once per workgroup, in the kernels that
// make their own operand terms).  The gate and the value are rounded as they would be
// stored, so the result has the bits of the product followed by the activation.
// 1024 -> 2 x 3072 -> 1024, both products (us): one row 11.6 -> 10.9 (a whole token, 28
// of them in 142 launches, shows no more than its spread); 16 rows 6.4 + 5.4 (fragments)
// + 5.9 -> 7.2 + 8.0; 2047 rows 70 + 14.2 + 44 -> 62 + 11.5 + 44.
__device__ __forceinline__ uint32_t proj_paired_tile(uint32_t pair, uint32_t t, uint32_t ntiles)
{
    return min(pair, ntiles / 2 - 1) + t * (ntiles / 2);         // (a pair past the end re-reads the last; dropped)
}

template <int ROWS = 8>
__device__ __forceinline__ void proj_store_pair(const ProjArgs& a, f32x4 gate, f32x4 value, uint32_t pair, uint32_t group,
                                                int lane, const float* scale = nullptr)
{
    const int c = lane & 15, g = lane >> 4;
    gate = proj_join_terms(gate);
    value = proj_join_terms(value);
    const uint32_t row = group * ROWS + (c & 7);
    if (c < ROWS && row < a.R && pair < a.N / 32) {
        const float sc = scale ? *scale : a.scales[row];
        f32x4 r;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float x = gate[i] * sc, y = value[i] * sc;
            asm volatile("" : "+v"(x), "+v"(y));                 // the products end here: no contraction into the activation
            r[i] = a.gate == kProjSrcGeglu ? proj_gated<kProjSrcGeglu>(x, y) : proj_gated<kProjSrcSwiglu>(x, y);
        }
        *reinterpret_cast<f32x4*>(a.y + (size_t)row * a.ldy + pair * 16 + g * 4) = r;
    }
}

// One row, a tile of eight gates (outputs 8 h .. 8 h + 7 of pair `pair`) and their values: lanes 32 and up hold the
// values' half.
__device__ __forceinline__ void proj_store_half_pair(const ProjArgs& a, f32x4 v, uint32_t pair, uint32_t h, int lane, float scale)
{
    v = proj_join_terms(v);
    f32x4 r;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        float x = v[i] * scale;
        asm volatile("" : "+v"(x));                              // (as above)
        const float y = wave_xor_f32(x, 32);
        r[i] = a.gate == kProjSrcGeglu ? proj_gated<kProjSrcGeglu>(x, y) : proj_gated<kProjSrcSwiglu>(x, y);
    }
    if ((lane & 47) == 0) *reinterpret_cast<f32x4*>(a.y + pair * 16 + h * 8 + (lane >> 4) * 4) = r;
}

// One wave-step: NT weight tiles against GROUPS operand fragments.
template <int GROUPS, int NT>
__device__ __forceinline__ void proj_step(f32x4 (&acc)[NT][GROUPS], const half8 (&wv)[NT],
                                          const half8* __restrict__ xp, uint32_t ktiles, uint32_t kt)
{
#pragma unroll
    for (int gi = 0; gi < GROUPS; gi++) {
        const half8 xb = xp[((size_t)gi * ktiles + kt) * 64];
#pragma unroll
        for (int t = 0; t < NT; t++)
            acc[t][gi] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv[t], xb, acc[t][gi], 0, 0, 0);
    }
}

// A wave's part of a product: NT tiles from nt0 on against all row groups, k-steps k_begin .. k_end - 1 in order.
template <int GROUPS, int NT, bool GATED>
__device__ __forceinline__ void proj_rows_sums(const ProjArgs& a, f32x4 (&acc)[NT][GROUPS], uint32_t nt0, uint32_t k_begin,
                                               uint32_t k_end, int lane)
{
    constexpr int KB = kProjKBatch / NT;                               // k-steps per register batch
    const uint32_t ktiles = a.K / 32, ntiles = a.N / 16;
    const half8* xp = a.xfrag + lane;
    // tile t of this wave; a run that sticks out past N re-reads the last tile and drops the result
    const half8* wp[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const uint32_t nt = GATED ? proj_paired_tile(nt0, t, ntiles) : (nt0 + t < ntiles) ? nt0 + t : ntiles - 1;
        wp[t] = a.w + (size_t)nt * ktiles * 64 + lane;
    }
    // W is read exactly once per launch (non-temporal); X fragments are
    // shared by every wave of the grid and stay cached.  Loads inside the
    // loop are unconditional and the last batch is peeled, so the
    // compiler's load counting keeps the prefetched batch in flight.
    half8 wa[KB][NT], wb[KB][NT];
    // The operand fragments travel a batch ahead with the weights: read when
    // needed they are cache hits, but a round trip to L2 per batch on a
    // chain of four to thirty batches that is the launch's critical path.
    half8 xa[KB][GROUPS], xb[KB][GROUPS];
    auto load_x = [&](half8 (&xv)[KB][GROUPS], uint32_t k0) {
#pragma unroll
        for (int u = 0; u < KB; u++)
#pragma unroll
            for (int gi = 0; gi < GROUPS; gi++) xv[u][gi] = xp[((size_t)gi * ktiles + k0 + u) * 64];
    };
    auto step = [&](const half8 (&wv)[NT], const half8 (&xv)[GROUPS]) {
#pragma unroll
        for (int gi = 0; gi < GROUPS; gi++)
#pragma unroll
            for (int t = 0; t < NT; t++)
                acc[t][gi] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv[t], xv[gi], acc[t][gi], 0, 0, 0);
    };
    uint32_t kt = k_begin;
    const uint32_t kper = k_end - k_begin;
    const uint32_t full_end = k_begin + kper / KB * KB;
    if (kt < full_end) {
#pragma unroll
        for (int u = 0; u < KB; u++)
#pragma unroll
            for (int t = 0; t < NT; t++)
                wa[u][t] = __builtin_nontemporal_load(&wp[t][(size_t)(kt + u) * 64]);
        load_x(xa, kt);
        while (kt + 2 * KB <= full_end) {
#pragma unroll
            for (int u = 0; u < KB; u++)
#pragma unroll
                for (int t = 0; t < NT; t++)
                    wb[u][t] = __builtin_nontemporal_load(&wp[t][(size_t)(kt + KB + u) * 64]);
            load_x(xb, kt + KB);
#pragma unroll
            for (int u = 0; u < KB; u++) step(wa[u], xa[u]);
#pragma unroll
            for (int u = 0; u < KB; u++) {
#pragma unroll
                for (int t = 0; t < NT; t++) wa[u][t] = wb[u][t];
#pragma unroll
                for (int gi = 0; gi < GROUPS; gi++) xa[u][gi] = xb[u][gi];
            }
            kt += KB;
        }
#pragma unroll
        for (int u = 0; u < KB; u++) step(wa[u], xa[u]);
        kt += KB;
    }
    for (; kt < k_end; kt++) {                               // part not a multiple of the batch
        half8 wv[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) wv[t] = __builtin_nontemporal_load(&wp[t][(size_t)kt * 64]);
        proj_step<GROUPS, NT>(acc, wv, xp, ktiles, kt);
    }
}

// GROUPS = row groups of eight (one or two), NT = 16-output tiles per wave
// (templates, so the accumulators stay in registers).  A workgroup is four
// waves.  With ksplit = 1 they own four consecutive runs of 16*NT outputs; with
// ksplit = 2 or 4 that many waves share a run and take contiguous parts of the
// input range (a narrow weight then still puts a thousand waves on the chip),
// and their sums are added through LDS in part order, so the result does not
// depend on timing.  Every X fragment a wave loads serves NT weight tiles:
// with two row groups (9..16 rows) NT = 2 keeps the operand traffic through
// the vector cache at the two bytes per weight byte of the one-group case.
template <int GROUPS, int NT, bool GATED = false>
__global__ __launch_bounds__(kProjThreads) void proj_rows_kernel(const ProjArgs a)
{
    static_assert(!GATED || NT == 2, "a gate's tile and a value's");
    // partial sums of the waves with part > 0: (4 / S) runs x (S - 1) parts <= 3 entries
    __shared__ f32x4 s_part[3 * NT * GROUPS * 64];

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t S = a.ksplit;
    const uint32_t slot = wave / S, part = wave % S;
    const uint32_t run = blockIdx.x * (4 / S) + slot;            // this wave's run of 16*NT outputs
    const uint32_t nt0 = GATED ? run : run * NT;                 // (GATED: a pair of tiles)
    const uint32_t ntiles = a.N / 16;
    const bool live = nt0 < (GATED ? ntiles / 2 : ntiles);                              // N/16 need not be a multiple of the runs per block
    const uint32_t ktiles = a.K / 32;
    const uint32_t kper = ktiles / S;                            // host guarantees divisibility
    const uint32_t k_begin = part * kper, k_end = k_begin + kper;

    f32x4 acc[NT][GROUPS];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int gi = 0; gi < GROUPS; gi++) acc[t][gi] = f32x4{0.f, 0.f, 0.f, 0.f};

    if (live) {
        proj_rows_sums<GROUPS, NT, GATED>(a, acc, nt0, k_begin, k_end, lane);
    }

    if (S > 1) {                                                 // uniform over the workgroup
        if (part > 0) {
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int gi = 0; gi < GROUPS; gi++)
                    s_part[(((slot * (S - 1) + (part - 1)) * NT + t) * GROUPS + gi) * 64 + lane] = acc[t][gi];
        }
        __syncthreads();
        if (part > 0) return;
        for (uint32_t p = 1; p < S; p++) {
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int gi = 0; gi < GROUPS; gi++) {
                    const f32x4 o = s_part[(((slot * (S - 1) + (p - 1)) * NT + t) * GROUPS + gi) * 64 + lane];
#pragma unroll
                    for (int i = 0; i < 4; i++) acc[t][gi][i] += o[i];
                }
        }
    }
    if (!live) return;

    if constexpr (GATED) {
#pragma unroll
        for (int gi = 0; gi < GROUPS; gi++) proj_store_pair(a, acc[0][gi], acc[1][gi], nt0, gi, lane);
        return;
    }
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int gi = 0; gi < GROUPS; gi++) proj_store_tile(a, acc[t][gi], nt0 + t, gi, lane);
}

// The product of 2 to 16 rows and a wide weight (ksplit = 1: the sums of proj_rows_kernel) into rows of page-locked host
// memory: the logits of a batched step, straight to where its sessions keep them.
//
// Bound by the link to the host: 16 rows of 151 936 are 9.7 MB, 175 us of it, against 66 for the weight from HBM (1024
// inputs).  A workgroup's 128 outputs pass through LDS and go out 512 bytes of a row at a time, and its place on the
// compute unit is free for the next one's weights while they travel.  The host gives a unit one workgroup (by its
// LDS), so that the first results are on the link after a fifth of the weight has been read, and not after all of it: 16
// rows, call to return, 216 us with all of 1187 workgroups at once, 205 so; 8 rows 133, 117; 2 rows 84, 78.  Against the
// product to device memory and rows_down_kernel behind it (us): 1024 -> 151 936, 2 / 4 / 8 / 16 rows 87 / 109 / 154 / 257
// -> 78 / 88 / 117 / 205; 2048 -> 65 536 70 / 79 / 98 / 141 -> 66 / 71 / 83 / 122; 4096 -> 32 768 70 / 73 / 83 / 101 ->
// 63 / 64 / 74 / 95.  A step of sixteen sessions 1.45 -> 1.39 ms.
struct ProjDownArgs {
    f32x4* y[16];
};

constexpr int kDownCols = 128, kDownStride = kDownCols + 4;

template <int GROUPS>
__global__ __launch_bounds__(kProjThreads) void proj_rows_down_kernel(const ProjArgs a, const ProjDownArgs d)
{
    constexpr int NT = 2;
    extern __shared__ __attribute__((aligned(16))) unsigned char down_smem[];
    float* stage = reinterpret_cast<float*>(down_smem);          // [8 GROUPS][kDownStride]
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t ntiles = a.N / 16, nt0 = (blockIdx.x * 4 + wave) * NT;
    f32x4* to[GROUPS];                                           // thread t: unit t % 32 of rows t / 32 + 8 gi
#pragma unroll
    for (int gi = 0; gi < GROUPS; gi++) to[gi] = d.y[min(gi * 8 + threadIdx.x / 32, a.R - 1)];
    f32x4 acc[NT][GROUPS];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int gi = 0; gi < GROUPS; gi++) acc[t][gi] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (nt0 < ntiles) proj_rows_sums<GROUPS, NT, false>(a, acc, nt0, 0, a.K / 32, lane);
    const int c = lane & 15, g = lane >> 4;
#pragma unroll
    for (int gi = 0; gi < GROUPS; gi++) {
        const float sc = a.scales[min((uint32_t)(gi * 8 + (c & 7)), a.R - 1)];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            f32x4 v = proj_join_terms(acc[t][gi]);
#pragma unroll
            for (int i = 0; i < 4; i++) v[i] *= sc;
            if (c < 8) *reinterpret_cast<f32x4*>(stage + (gi * 8 + c) * kDownStride + (wave * NT + t) * 16 + g * 4) = v;
        }
    }
    lds_barrier();
    const uint32_t unit = threadIdx.x % 32, at = blockIdx.x * (kDownCols / 4) + unit;
    if (at >= a.N / 4) return;
#pragma unroll
    for (int gi = 0; gi < GROUPS; gi++) {
        const uint32_t row = gi * 8 + threadIdx.x / 32;
        if (row < a.R) to[gi][at] = *reinterpret_cast<const f32x4*>(stage + row * kDownStride + unit * 4);
    }
}

// One row (a decode step): proj_rows_kernel<1, 1> with the fragment kernel
// folded in.  Every workgroup builds the row's operand terms in its own LDS
// (4 bytes per input: hi and lo of the one live column pair) while its first
// batches of weights are on the way, instead of reading fragments a launch before
// it wrote: a decode step is a chain of dependent launches of a few
// microseconds each, and this removes four of ten per layer.  The row's values,
// the scale and the order of every sum are those of proj_prep_kernel followed
// by proj_rows_kernel<1, 1> (same helpers, same loops), so the result has the
// same bits: a serial step still equals its row of a batched step.
//
// Order of the requests: the row (with the norm's weights, the gate's partner
// values and the residual) FIRST, then up to three batches of weights (24
// k-steps: the whole share of a wave for inputs up to 3072 at four waves per
// tile).  A wave's loads come back in the order they were asked for, so a row
// asked for after the weights is not there before them (2.0 us after the
// workgroup's start, measured, against 0.8); asked for first, the sums over the
// row run while the weights travel.  NB0 = batches asked for up front, a
// template parameter so that every load before the first wait is unconditional
// and the compiler's count of loads in flight is exact.
//
// FORM: kRow1Gated takes the gates' tile and the values' (KB = 4 k-steps of both to a
// batch), and half as many workgroups as the plain form.  kRow1GatedHalf takes eight
// gates and their eight values as one tile, so a workgroup reads what a plain one does,
// in pieces of a line; for products whose pairs would leave half the CUs without a
// workgroup (whole FFNs of one row, us: 4096 -> 2 x 1024 11.4, against 13.3 of pairs and
// 11.3 of products that keep gates and values apart; 1024 -> 2 x 1024 8.2, 8.6, 7.6; 1056
// -> 2 x 4096 14.0, 15.8, 14.0; from 2 x 2560 on pairs are the faster: 4096 -> 18.0, 19.0
// apart).
constexpr int kRow1Plain = 0, kRow1Gated = 1, kRow1GatedHalf = 2;

template <int SRC, int NB0, int FORM, int KB>
__device__ __forceinline__ void proj_row1_body(const ProjArgs& a, const ProjPrepArgs& p, half8* sfrag,
                                               f32x4* s_part, float* s4, float* s_scale)
{
    constexpr bool GATED = FORM == kRow1Gated, HALF = FORM == kRow1GatedHalf;
    constexpr int NT = GATED ? 2 : 1;                            // weight tiles of a wave
    constexpr int CH = 2;                                        // chunks of eight inputs a thread can hold
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t t = threadIdx.x;
    const uint32_t S = a.ksplit;
    const uint32_t slot = wave / S, part = wave % S;
    const uint32_t nt0 = blockIdx.x * (4 / S) + slot;
    const uint32_t ntiles = a.N / 16;
    const bool live = nt0 < (GATED ? ntiles / 2 : ntiles);       // (GATED: nt0 is a pair of tiles, HALF: half a pair)
    const uint32_t ktiles = a.K / 32, nchunks = a.K / 8;
    const uint32_t kper = ktiles / S;
    const uint32_t k_begin = part * kper, k_end = k_begin + kper;
    const half8* wp[NT];
#pragma unroll
    for (int tt = 0; tt < NT; tt++)
        wp[tt] = a.w + (size_t)(GATED ? proj_paired_tile(nt0, tt, ntiles) : live ? nt0 : ntiles - 1) * ktiles * 64 + lane;
    if constexpr (HALF)      // rows 8 h .. 8 h + 7 of the gates' tile, then of the values'
        wp[0] = a.w + (size_t)proj_paired_tile(nt0 / 2, (lane >> 3) & 1, ntiles) * ktiles * 64 + (lane & 48) + nt0 % 2 * 8 + (lane & 7);
    const float* xr = p.x;
    const bool in_regs = a.K <= 2048u * CH;                      // uniform

    // 1. the row and what goes with it (a chunk past the end re-reads the last one; dropped below)
    f32x4 xl[CH], xh[CH];
    f32x4 el[SRC == kProjSrcPlain ? 1 : CH], eh[SRC == kProjSrcPlain ? 1 : CH];     // norm weights / gate partners
    if (in_regs) {
#pragma unroll
        for (int i = 0; i < CH; i++) {
            const uint32_t qc = min(t + 256u * i, nchunks - 1);
            xl[i] = *reinterpret_cast<const f32x4*>(xr + qc * 8);
            xh[i] = *reinterpret_cast<const f32x4*>(xr + qc * 8 + 4);
            if constexpr (SRC == kProjSrcRmsNorm) {
                el[i] = *reinterpret_cast<const f32x4*>(p.norm_w + qc * 8);
                eh[i] = *reinterpret_cast<const f32x4*>(p.norm_w + qc * 8 + 4);
            } else if constexpr (SRC == kProjSrcSwiglu || SRC == kProjSrcGeglu) {
                el[i] = *reinterpret_cast<const f32x4*>(xr + a.K + qc * 8);
                eh[i] = *reinterpret_cast<const f32x4*>(xr + a.K + qc * 8 + 4);
            }
        }
    }

    // 1b. the residual values the store at the very end will add, for every lane
    // and whether or not there is a residual (the row's start stands in): a load
    // that is only sometimes issued would turn the exact waits below into waits
    // for everything in flight
    f32x4 resid;
    {
        const int rc = lane & 15, rg = lane >> 4;
        const uint32_t rrow = min((uint32_t)(rc & 7), a.R - 1), rnt = min(nt0, ntiles - 1);
        const float* rp = a.bias_rows ? a.bias_rows + (size_t)rrow * a.ldy + rnt * 16 + rg * 4 : xr + rg * 4;
        resid = *reinterpret_cast<const f32x4*>(rp);
    }

    // 2. the weights: NB0 batches now, the rest as the buffers come free
    half8 wa[KB][NT], wb[KB][NT], wc[KB][NT];
    const uint32_t nb = kper / KB;                               // whole batches of this wave (>= NB0)
    auto load_batch = [&](half8 (&w)[KB][NT], uint32_t b) {
#pragma unroll
        for (int u = 0; u < KB; u++)
#pragma unroll
            for (int tt = 0; tt < NT; tt++)
                w[u][tt] = __builtin_nontemporal_load(&wp[tt][(size_t)(k_begin + b * KB + u) * 64]);
    };
    if constexpr (NB0 > 0) load_batch(wa, 0);
    if constexpr (NB0 > 1) load_batch(wb, 1);
    if constexpr (NB0 > 2) load_batch(wc, 2);

    // 3. the row's terms, as proj_prep_kernel forms them
    auto put_chunk = [&](uint32_t q, const float (&v)[8], float inv) {
        half8 hi, lo;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const float sv = v[j] * inv;
            _Float16 h = (_Float16)sv;
            if (fabsf((float)h) < 6.103515625e-05f) h = (_Float16)0.0f;      // 2^-14
            hi[j] = h;
            lo[j] = (_Float16)((sv - (float)h) * kProjLoScale);
        }
        sfrag[q * 2] = hi;
        sfrag[q * 2 + 1] = lo;
    };
    if (in_regs) {
        // One read of the row: its values stay in registers between the passes
        // (sum of squares, largest magnitude, terms).  Same values, same order of
        // the sum as the passes of the other branch (thread t takes the chunks t,
        // t + 256, ... in order).
        float v[CH][8];
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < CH; i++) {
            const bool has = t + 256u * i < nchunks;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                v[i][j] = has ? xl[i][j] : 0.f;
                v[i][4 + j] = has ? xh[i][j] : 0.f;
            }
            if constexpr (SRC == kProjSrcRmsNorm) {
#pragma unroll
                for (int j = 0; j < 8; j++) ss = fmaf(v[i][j], v[i][j], ss);
            }
        }
        if constexpr (SRC == kProjSrcRmsNorm) {
            const float inv_rms = 1.0f / sqrtf(block_sum_256(ss, s4) / (float)a.K + p.eps);
#pragma unroll
            for (int i = 0; i < CH; i++) {
                if (t + 256u * i < nchunks) {
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        v[i][j] = v[i][j] * inv_rms * el[i][j];
                        v[i][4 + j] = v[i][4 + j] * inv_rms * eh[i][j];
                    }
                }
            }
        } else if constexpr (SRC == kProjSrcSwiglu || SRC == kProjSrcGeglu) {
#pragma unroll
            for (int i = 0; i < CH; i++) {
                if (t + 256u * i < nchunks) {
#pragma unroll
                    for (int j = 0; j < 8; j++) v[i][j] = proj_gated<SRC>(v[i][j], j < 4 ? el[i][j] : eh[i][j - 4]);
                }
            }
        }
        float mx = 0.f;
#pragma unroll
        for (int i = 0; i < CH; i++)
#pragma unroll
            for (int j = 0; j < 8; j++) mx = fmaxf(mx, fabsf(v[i][j]));
        mx = block_max_256(mx, s4 + 4);
        uint32_t ex = (__float_as_uint(mx) >> 23) & 0xFFu;
        if (ex == 0 || ex == 0xFF) ex = 127;
        if (ex > 253) ex = 253;
        if (t == 0) *s_scale = __uint_as_float(ex << 23);
        const float inv = __uint_as_float((254u - ex) << 23);
#pragma unroll
        for (int i = 0; i < CH; i++) {
            const uint32_t q = t + 256u * i;
            if (q < nchunks) put_chunk(q, v[i], inv);
        }
    } else {
        float inv_rms = 1.0f;
        if constexpr (SRC == kProjSrcRmsNorm)
            inv_rms = 1.0f / sqrtf(row_sumsq_256(xr, a.K, s4) / (float)a.K + p.eps);
        float mx = 0.f;
        for (uint32_t k = t; k < a.K; k += 256) mx = fmaxf(mx, fabsf(proj_src_value<SRC>(p, xr, k, inv_rms)));
        mx = block_max_256(mx, s4 + 4);
        uint32_t ex = (__float_as_uint(mx) >> 23) & 0xFFu;
        if (ex == 0 || ex == 0xFF) ex = 127;
        if (ex > 253) ex = 253;
        if (t == 0) *s_scale = __uint_as_float(ex << 23);
        const float inv = __uint_as_float((254u - ex) << 23);
        for (uint32_t q = t; q < nchunks; q += 256) {
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = proj_src_value<SRC>(p, xr, q * 8 + j, inv_rms);
            put_chunk(q, v, inv);
        }
    }
    lds_barrier();                                              // the terms are in LDS (the weights may still be on their way)

    // B operand of k-step kt: column 0 = hi, column 8 = lo of row 0, the rest zero
    const int c = lane & 15, g = lane >> 4;
    const bool has = (c & 7) == 0;
    const half8* my = sfrag + g * 2 + (c >> 3);
    half8 zero;
#pragma unroll
    for (int j = 0; j < 8; j++) zero[j] = (_Float16)0.0f;
    f32x4 acc[NT];
#pragma unroll
    for (int tt = 0; tt < NT; tt++) acc[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto step = [&](const half8 (&wv)[NT], uint32_t k) {
        const half8 xb = has ? my[(size_t)k * 8] : zero;
#pragma unroll
        for (int tt = 0; tt < NT; tt++) acc[tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv[tt], xb, acc[tt], 0, 0, 0);
    };
    // k-steps in ascending order, whatever buffer holds them (the order of the sum
    // is that of proj_rows_kernel<1, 1>)
    auto steps = [&](const half8 (&w)[KB][NT], uint32_t b) {
#pragma unroll
        for (int u = 0; u < KB; u++) step(w[u], k_begin + b * KB + u);
    };
    if constexpr (NB0 > 0) {
        steps(wa, 0);
        if (NB0 > 2 && nb > 3) load_batch(wa, 3);
    }
    if constexpr (NB0 > 1) {
        steps(wb, 1);
        if (NB0 > 2 && nb > 4) load_batch(wb, 4);
    }
    if constexpr (NB0 > 2) {
        steps(wc, 2);
        for (uint32_t b = 3; b < nb; b += 2) {                   // wa holds batch b, wb batch b + 1
            steps(wa, b);
            if (b + 2 < nb) load_batch(wa, b + 2);
            if (b + 1 < nb) {
                steps(wb, b + 1);
                if (b + 3 < nb) load_batch(wb, b + 3);
            }
        }
    }
    for (uint32_t kt = k_begin + nb * KB; kt < k_end; kt++) {
        half8 wv[NT];
#pragma unroll
        for (int tt = 0; tt < NT; tt++) wv[tt] = __builtin_nontemporal_load(&wp[tt][(size_t)kt * 64]);
        step(wv, kt);
    }

    if (S > 1) {                                                 // uniform over the workgroup
        if (part > 0) {
#pragma unroll
            for (int tt = 0; tt < NT; tt++) s_part[((slot * (S - 1) + (part - 1)) * NT + tt) * 64 + lane] = acc[tt];
        }
        __syncthreads();
        if (part > 0) return;
        for (uint32_t pp = 1; pp < S; pp++) {
#pragma unroll
            for (int tt = 0; tt < NT; tt++) {
                const f32x4 o = s_part[((slot * (S - 1) + (pp - 1)) * NT + tt) * 64 + lane];
#pragma unroll
                for (int i = 0; i < 4; i++) acc[tt][i] += o[i];
            }
        }
    }
    if (!live) return;
    if constexpr (GATED)
        proj_store_pair(a, acc[0], acc[1], nt0, 0, lane, s_scale);
    else if constexpr (HALF)
        proj_store_half_pair(a, acc[0], nt0 / 2, nt0 % 2, lane, *s_scale);
    else
        proj_store_tile(a, acc[0], nt0, 0, lane, s_scale, &resid);
}

// LDS of proj_row1_kernel beside the row's terms: partial tiles, the row's sums, its scale.
constexpr size_t row1_static_lds(bool gated) { return (gated ? 6 : 3) * 64 * sizeof(f32x4) + 8 * sizeof(float) + sizeof(float); }

template <int SRC, int FORM = kRow1Plain>
__global__ __launch_bounds__(kProjThreads) void proj_row1_kernel(const ProjArgs a, const ProjPrepArgs p)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char row1_smem[];
    half8* sfrag = reinterpret_cast<half8*>(row1_smem);           // [K/8][2]: hi, lo of chunk q
    __shared__ f32x4 s_part[(FORM == kRow1Gated ? 6 : 3) * 64];
    __shared__ float s4[8];
    __shared__ float s_scale;
    const uint32_t kper = a.K / 32 / a.ksplit;                    // a wave's k-steps; whole batches of KB: uniform
    const auto body = [&](auto batch) {
        constexpr int KB = decltype(batch)::value;
        const uint32_t nb = kper / KB;
        if (nb >= 3)
            proj_row1_body<SRC, 3, FORM, KB>(a, p, sfrag, s_part, s4, &s_scale);
        else if (nb == 2)
            proj_row1_body<SRC, 2, FORM, KB>(a, p, sfrag, s_part, s4, &s_scale);
        else if (nb == 1)
            proj_row1_body<SRC, 1, FORM, KB>(a, p, sfrag, s_part, s4, &s_scale);
        else
            proj_row1_body<SRC, 0, FORM, KB>(a, p, sfrag, s_part, s4, &s_scale);
    };
    if (FORM == kRow1Gated || (FORM == kRow1GatedHalf && kper % kProjKBatch))
        body(std::integral_constant<int, kProjKBatch / 2>());
    else
        body(std::integral_constant<int, kProjKBatch>());
}

// Two rows to a few dozen, inputs of 512 D / 4: the fragment step inside the product.
// A batched decode step is a chain of short launches, and of its nine per layer four
// only wrote fragments (4.6 us each, 16 workgroups).  Here a workgroup, NT tiles of 16
// outputs by a row group, makes the fragments of its eight rows itself: every wave
// those of its own quarter of the inputs, in LDS nobody else reads, while its whole
// share of the weights is on the way (D x NT KiB in registers).  The rows are asked
// for first (a wave's loads come back in order).  Bound by latency, and by the vector
// ALU time of the terms, which is the same however many outputs a workgroup has: the
// host gives a CU one workgroup.  Values, scale, the order of the norm's sum and the
// order of the product's are those of proj_prep_kernel and of the kernels that share a
// tile's inputs between four waves, so the result has the same bits.
//
// A workgroup of ROWS = 8 rows fills the operand's columns; one of four leaves half of them unused and has half the
// terms to make, for narrow weights whose tiles of eight rows leave compute units without work.  Eight rows / four
// (us, weights from HBM, plain rows): 16 rows, 3072 -> 1024 7.8 / 5.7, 2048 -> 1024 5.5 / 4.2, 1536 -> 512 4.6 / 3.7,
// norm + 1024 -> 1024 4.5 / 3.6; 8 rows, 2048 -> 2048 5.6 / 4.7; 4 rows, norm + 1024 -> 4096 4.2 / 3.8; 1024 -> 1024
// at any number of rows 3.7 / 3.7.
//
// 16 rows, weights from HBM, against proj_prep_kernel + proj_gemm_split_kernel<1, 1, 8>
// (us): norm + 1024 -> 4096 8.1 -> 5.2, norm + 1024 -> 6144 9.3 -> 6.2, 2048 -> 1024
// 7.7 -> 5.5 -> 4.2, 3072 -> 1024 9.5 -> 7.8 -> 5.7; 32 rows of the third 7.8 -> 5.5.  (A lane making
// the terms of four inputs of its own operand column and trading them with the lane
// eight on, no LDS: 5.7, 6.7, 5.8, 8.1.)
template <int SRC, int D, int NT, bool GATED = false, int ROWS = 8>
__global__ __launch_bounds__(kProjThreads, 1) void proj_rows_fused_kernel(const ProjArgs a, const ProjPrepArgs p)
{
    static_assert(D % 2 == 0 && (SRC == kProjSrcPlain || (SRC == kProjSrcRmsNorm && D <= 16)), "sources held in registers");
    static_assert(ROWS == 8 || ROWS == 4, "operand columns: hi terms 0 .. ROWS - 1, lo terms eight on");
    static_assert(!GATED || NT % 2 == 0, "gates' tiles and values'");
    constexpr bool NORM = SRC == kProjSrcRmsNorm;
    constexpr int KT = 4 * D;                                    // k-steps of a row
    constexpr int QS = 16 / ROWS;                                // k-steps that the lanes of a wave span
    constexpr int CH = D / QS;                                   // chunks of eight inputs per lane
    static_assert(D % QS == 0, "whole spans");
    extern __shared__ __attribute__((aligned(16))) unsigned char fused_smem[];
    // sums of squares of the chunks, by row, chunk of a k-step and k-step
    __shared__ __attribute__((aligned(16))) float s_ss[NORM ? ROWS : 1][NORM ? 4 : 1][NORM ? KT + 4 : 1];
    __shared__ float s_mx[4][ROWS];
    __shared__ f32x4 s_red[3 * NT * 64];
    const int lane = threadIdx.x & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t ntiles = a.N / 16, nt0 = blockIdx.x * NT, group = blockIdx.y;
    const uint32_t k0 = wave * D;                                // this wave's quarter of the k-steps
    half8* frag = reinterpret_cast<half8*>(fused_smem) + k0 * 64;

    // 1. the rows, what goes with them, then the weights, all at once.  A lane takes chunk lane / ROWS of every QS k-steps
    // of row lane % ROWS: eight lanes read 256 bytes of a row, sixteen 512.  (A row past the end re-reads the last; its columns are dropped.)
    const uint32_t r = lane % ROWS, q = lane / ROWS;
    const uint32_t at = k0 * 32 + q * 8;
    const float* xr = p.x + (size_t)min(group * ROWS + r, a.R - 1) * p.ldx + at;
    f32x4 x[CH][2], nw[NORM ? CH : 1][2];
#pragma unroll
    for (int i = 0; i < CH; i++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
            x[i][h] = *reinterpret_cast<const f32x4*>(xr + i * QS * 32 + h * 4);
            if constexpr (NORM) nw[i][h] = *reinterpret_cast<const f32x4*>(p.norm_w + at + i * QS * 32 + h * 4);
        }
    f32x4 resid[NT];
    half8 w[D][NT];
    const half8* wp[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const uint32_t tile = GATED ? proj_paired_tile((nt0 + t) / 2, t % 2, ntiles) : min(nt0 + t, ntiles - 1);   // (one past the end: dropped)
        const uint32_t row = min(group * ROWS + lane % ROWS, a.R - 1);
        resid[t] = *reinterpret_cast<const f32x4*>(
            !GATED && a.bias_rows ? a.bias_rows + (size_t)row * a.ldy + tile * 16 + (lane >> 4) * 4 : xr);
        wp[t] = a.w + ((size_t)tile * KT + k0) * 64;
    }
#pragma unroll
    for (int u = 0; u < D; u++)
#pragma unroll
        for (int t = 0; t < NT; t++) w[u][t] = wp[t][u * 64 + lane];

    // 2. the rows' norms: every chunk of eight summed in order, the chunks by the tree of block_sum_256
    if constexpr (NORM) {
#pragma unroll
        for (int i = 0; i < CH; i++) {
            float ss = 0.f;
#pragma unroll
            for (int j = 0; j < 8; j++) ss = fmaf(x[i][j / 4][j % 4], x[i][j / 4][j % 4], ss);
            s_ss[r][q & 3][k0 + QS * i + (q >> 2)] = ss;
        }
        lds_barrier();
        // of 64 chunks = 16 k-steps: bits 5 .. 2 of a chunk's number are the k-step's, added in registers; bits 1 and 0
        // the chunk of the k-step, which lanes ROWS r' + r hold (q & 3 here, so that the lanes 2 ROWS and ROWS on have the others)
        float part[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < (KT + 15) / 16; j++) {
            float v[16];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                f32x4 four = f32x4{0.f, 0.f, 0.f, 0.f};
                if (16 * j + 4 * i < KT) four = *reinterpret_cast<const f32x4*>(&s_ss[r][q & 3][16 * j + 4 * i]);
#pragma unroll
                for (int e = 0; e < 4; e++) v[4 * i + e] = four[e];
            }
#pragma unroll
            for (int half = 8; half >= 1; half /= 2)
#pragma unroll
                for (int i = 0; i < half; i++) v[i] += v[i + half];
            v[0] += wave_xor_f32(v[0], 2 * ROWS);
            part[j] = v[0] + wave_xor_f32(v[0], ROWS);
        }
        const float inv_rms = 1.0f / sqrtf(((part[0] + part[1]) + (part[2] + part[3])) / (float)a.K + p.eps);
#pragma unroll
        for (int i = 0; i < CH; i++)
#pragma unroll
            for (int j = 0; j < 8; j++) x[i][j / 4][j % 4] = x[i][j / 4][j % 4] * inv_rms * nw[i][j / 4][j % 4];
    }

    // 3. the rows' scales
    float mx = 0.f;
#pragma unroll
    for (int i = 0; i < CH; i++)
#pragma unroll
        for (int j = 0; j < 8; j++) mx = fmaxf(mx, fabsf(x[i][j / 4][j % 4]));
#pragma unroll
    for (int off = ROWS; off < 64; off *= 2) mx = fmaxf(mx, wave_xor_f32(mx, off));
    if (lane < ROWS) s_mx[wave][lane] = mx;
    lds_barrier();
    mx = fmaxf(fmaxf(s_mx[0][r], s_mx[1][r]), fmaxf(s_mx[2][r], s_mx[3][r]));
    uint32_t ex = (__float_as_uint(mx) >> 23) & 0xFFu;
    if (ex == 0 || ex == 0xFF) ex = 127;
    if (ex > 253) ex = 253;
    const float scale = __uint_as_float(ex << 23), inv = __uint_as_float((254u - ex) << 23);

    // 4. the terms, into this wave's own fragments (no barrier: a wave's LDS accesses stay in order), and the product
    f32x4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < CH; i++) {
        half8 hi, lo;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            // (proj_write_chunk's terms in fewer instructions: (s - h) 2^11 and s 2^11 - h 2^11 are both exact)
            const float sv = x[i][j / 4][j % 4] * inv;
            _Float16 h = (_Float16)sv;
            if (__builtin_fabsf16(h) < (_Float16)6.103515625e-05f) h = (_Float16)0.0f;      // 2^-14
            hi[j] = h;
            lo[j] = (_Float16)fmaf((float)h, -kProjLoScale, sv * kProjLoScale);
        }
        half8* to = frag + (QS * i + (q >> 2)) * 64 + 16 * (q & 3) + r;
        to[0] = hi;
        to[8] = lo;
    }
#pragma unroll
    for (int u = 0; u < D; u++) {
        const half8 xb = frag[u * 64 + (lane & ~(8 - ROWS))];   // (ROWS = 4: columns 4 on are copies, dropped)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[u][t], xb, acc[t], 0, 0, 0);
    }

    // 5. the waves' parts, in order
    if (wave > 0) {
#pragma unroll
        for (int t = 0; t < NT; t++) s_red[((wave - 1) * NT + t) * 64 + lane] = acc[t];
    }
    lds_barrier();
    if (wave > 0) return;
#pragma unroll
    for (int t = 0; t < NT; t++) {
#pragma unroll
        for (int part = 0; part < 3; part++) {
            const f32x4 other = s_red[(part * NT + t) * 64 + lane];
#pragma unroll
            for (int i = 0; i < 4; i++) acc[t][i] += other[i];
        }
        if constexpr (!GATED)
            proj_store_tile<ROWS>(a, acc[t], nt0 + t, group, lane, &scale, &resid[t]);
        else if (t % 2 == 1)
            proj_store_pair<ROWS>(a, acc[t - 1], acc[t], (nt0 + t) / 2, group, lane, &scale);
    }
}

// Products too small to fill the chip with the LDS-staged tiles below, from two
// rows on: a register-tiled GEMM on the same two layouts.  The four waves of a
// workgroup share one tile of NT x GROUPS accumulator tiles (16 NT outputs x
// 8 GROUPS rows) and take a quarter of the input range each; their sums meet in
// LDS and are added in wave order, each wave adding and storing every fourth tile.
// Every k-step loads NT weight tiles and GROUPS operand fragments, one KiB each and
// both already in operand order, and feeds NT x GROUPS MFMAs.  These products are
// bound by load latency (the weights come from HBM, a few MB, one to three
// microseconds of it) and, as the rows grow, by the bytes that pass the vector
// cache, so a wave keeps D k-steps on their way: eight of a small tile are the
// whole share of a wave at 1024 inputs.  Loads stand behind the MFMAs that free
// their registers; in whole turns of D none is conditional, so the compiler's count
// of loads in flight is exact, and what is left behind the last turn is asked for all
// at once (in registers of its own name: kept in those of the turns, the compiler
// holds both; one after the other, 8 rows of 896 -> 4096 took 8.0 us, 6.3 now).
// grid.x walks the outputs,
// so the workgroups the dispatcher deals round-robin to the eight XCDs differ in
// output tile.
//
// Measured (us, weights from HBM; one k-step ahead, tiles <4, 2>, as this kernel
// was, against <2, 1, 8> (<1, 1, 8> for 1024 outputs) at 20 and 45 rows, <2, 2, 8> at
// 100 and 200, <4, 2, 4> at 511):
//   rows            20           45           100          200          511
//   1024 -> 4096    8.4 / 4.8    8.7 / 6.0    9.8 / 8.5    13.2 / 12.2  (LDS tiles)
//   3072 -> 1024   15.1 / 5.5   15.4 / 6.7   15.3 / 8.0    15.7 / 11.5  20.4 / 19.3
// (Below 64 rows a kernel of one wave per 64 outputs x 32 rows ran before: 20 us
// for the first, 51 for the second.)  Eight waves to the input range, or deeper
// turns on larger tiles, gave nothing.
template <int GROUPS, int NT, int D, bool GATED = false>
__global__ __launch_bounds__(kProjThreads, GROUPS * NT == 8 ? 3 : 2) void proj_gemm_split_kernel(const ProjArgs a)
{
    __shared__ f32x4 s_red[4 * NT * GROUPS * 64];
    const int lane = threadIdx.x & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t ktiles = a.K / 32, ntiles = a.N / 16, ngroups = (a.R + 7) / 8;
    const uint32_t nt0 = blockIdx.x * NT, group0 = blockIdx.y * GROUPS;
    const uint32_t k_begin = ktiles * wave / 4, n = ktiles * (wave + 1) / 4 - k_begin;   // (none: a wave adds zeros)

    // a tile or group past the end re-reads the last one; its result is dropped
    const half8* wp[NT];
    const half8* xp[GROUPS];
#pragma unroll
    for (int t = 0; t < NT; t++)
        wp[t] = a.w + ((size_t)(GATED ? proj_paired_tile((nt0 + t) / 2, t % 2, ntiles) : min(nt0 + t, ntiles - 1)) * ktiles + k_begin) * 64;
#pragma unroll
    for (int gi = 0; gi < GROUPS; gi++)
        xp[gi] = a.xfrag + ((size_t)min(group0 + gi, ngroups - 1) * ktiles + k_begin) * 64;

    f32x4 acc[NT][GROUPS];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int gi = 0; gi < GROUPS; gi++) acc[t][gi] = f32x4{0.f, 0.f, 0.f, 0.f};

    half8 w[D][NT], x[D][GROUPS];
    auto load_set = [&](half8 (&wv)[NT], half8 (&xv)[GROUPS], uint32_t k) {
        const uint32_t o = k * 64 + lane;
#pragma unroll
        for (int t = 0; t < NT; t++) wv[t] = wp[t][o];
#pragma unroll
        for (int gi = 0; gi < GROUPS; gi++) xv[gi] = xp[gi][o];
    };
    auto mfma_set = [&](const half8 (&wv)[NT], const half8 (&xv)[GROUPS]) {
#pragma unroll
        for (int gi = 0; gi < GROUPS; gi++)
#pragma unroll
            for (int t = 0; t < NT; t++)
                acc[t][gi] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv[t], xv[gi], acc[t][gi], 0, 0, 0);
    };
    const uint32_t turns = n / D, rest = n - turns * D;
    if (turns) {
#pragma unroll
        for (int d = 0; d < D; d++) load_set(w[d], x[d], d);
        for (uint32_t turn = 1; turn < turns; turn++) {
#pragma unroll
            for (int d = 0; d < D; d++) {
                mfma_set(w[d], x[d]);
                load_set(w[d], x[d], turn * D + d);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int d = 0; d < D; d++) mfma_set(w[d], x[d]);
    }
    if (__builtin_expect(rest != 0, 0)) {
        half8 wr[D - 1][NT], xr[D - 1][GROUPS];
#pragma unroll
        for (int d = 0; d < D - 1; d++)
            if ((uint32_t)d < rest) load_set(wr[d], xr[d], turns * D + d);
#pragma unroll
        for (int d = 0; d < D - 1; d++)
            if ((uint32_t)d < rest) mfma_set(wr[d], xr[d]);
    }

#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int gi = 0; gi < GROUPS; gi++) s_red[((wave * NT + t) * GROUPS + gi) * 64 + lane] = acc[t][gi];
    lds_barrier();
    auto sum = [&](uint32_t i) {
        f32x4 v = s_red[i * 64 + lane];
#pragma unroll
        for (int p = 1; p < 4; p++) {
            const f32x4 o = s_red[(p * NT * GROUPS + i) * 64 + lane];
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] += o[j];
        }
        return v;
    };
    if constexpr (GATED) {
        static_assert(NT % 2 == 0, "gates' tiles and values'");
#pragma unroll 1
        for (uint32_t i = wave; i < NT / 2 * GROUPS; i += 4) {
            const uint32_t pair = i / GROUPS, gi = i % GROUPS;
            proj_store_pair(a, sum(2 * pair * GROUPS + gi), sum((2 * pair + 1) * GROUPS + gi), nt0 / 2 + pair, group0 + gi, lane);
        }
    } else {
#pragma unroll 1
        for (uint32_t i = wave; i < NT * GROUPS; i += 4)
            proj_store_tile(a, sum(i), nt0 + i / GROUPS, group0 + i % GROUPS, lane);
    }
}

// Many rows, products that fill the chip with 128-output x 128-row workgroup
// tiles (2 x 2 waves of 64 x 64): operands staged through LDS.  Per k-step the
// workgroup needs 8 weight tiles and 16 operand fragments, 24 KiB that are
// already in operand order: every wave copies six of them with direct-to-LDS
// loads (no registers, so the copies run two k-steps ahead of the MFMAs in a
// ring of three stages), and reads the 4 + 8 KiB of its own wave tile back with
// 128-bit LDS reads, lane i at 16 i: conflict free.  Against loading the wave
// tile's operands into registers directly the vector cache moves half the
// bytes per MFMA and the prefetch depth costs no registers.  grid.x walks the
// output panels, so one XCD's L2 holds an eighth of the weight and all of the
// fragments.
//
// Step kt: wait for this wave's copies of stage kt (the six of stage kt + 1 may
// still be in flight), workgroup barrier (everybody's copies of stage kt have
// landed, and everybody has finished reading stage kt - 1), start the copies
// of stage kt + 2 into the slot of stage kt - 1, then read and multiply.
//
// GROUPS = 8 is the tile described above; GROUPS = 4 halves the rows (128
// outputs x 64 rows, 16 KiB per stage) for products with too few rows to fill
// the chip with the large one.
// WN = waves side by side along the outputs (2 or 4; two wave rows always),
// RING = stages.  <8, 2, 3>: the tile above.  <4, 2, 3>: 128 x 64 for products
// with too few rows to fill the chip with the large one.  <8, 4, 5>: eight
// waves, 256 outputs x 128 rows, 32 KiB per stage copied four k-steps ahead,
// one workgroup per CU: a third fewer bytes per MFMA than the four-wave tile.
template <int GROUPS, int WN, int RING, int KS = 1>
constexpr size_t gemm_lds_bytes()
{
    return (size_t)KS * RING * (WN * 4 + 2 * GROUPS) * 1024;   // KiB per stage and set of waves: 4 WN weight tiles, 2 GROUPS fragments
}

// PIPE: the operand reads of the next k-step are issued before this one's MFMAs
// (two register sets), for launches that leave a SIMD with a single wave and
// nobody else to cover its LDS latency; needs one more ring stage, because a
// stage is now read one k-step before it is used.  With five stages one barrier does for two
// k-steps.  A step goes by quarters (copies and reads among the MFMAs).  us, before / now, operand
// fragments included: 2047 rows, 1024 -> 4096 in <8, 4, 5> 54.1 / 51.7 (read behind a barrier a step in <8, 4, 4>
// before), 4095 rows gated 1024 -> 2 x 3072 120.7 / 115.3; in <4, 2, 4> with two sets of waves 2047 rows 2048 -> 1024 33.0 / 31.9, 3072 ->
// 1024 43.3 / 41.3.
//
// KS = 2: two such sets of waves in one workgroup, each with its own ring, take
// one half of the input range each (the host asks for it only when the number of
// k-steps is even); the upper half's sums pass through LDS at the end and the
// lower half adds them to its own, always in that order.  For products whose
// tiles give every CU one workgroup and no more (a SIMD would hold a single wave
// for a long chain of k-steps): twice the waves per SIMD, half the chain.
template <int GROUPS, int WN, int RING, bool PIPE = false, int KS = 1, bool GATED = false>
__global__ __launch_bounds__(128 * WN * KS, (WN == 2 && KS == 1) ? 2 : 1) void proj_gemm_lds_kernel(const ProjArgs a)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char gemm_smem[];
    constexpr int NT = 4, WAVES = 2 * WN, CHUNKS = WN * NT + 2 * GROUPS, CPW = CHUNKS / WAVES;
    static_assert(CHUNKS % WAVES == 0, "every wave copies the same number of chunks");
    static_assert(KS == 1 || KS == 2, "one set of waves, or two that halve the input range");
    constexpr uint32_t STAGE = CHUNKS * 1024;
    const int lane = threadIdx.x & 63;
    const uint32_t wave_wg = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t kh = wave_wg / WAVES, wave = wave_wg % WAVES;      // half of the input range, wave of the set
    const uint32_t wn = wave % WN, wr = wave / WN;
    const uint32_t ktiles_row = a.K / 32, ntiles = a.N / 16, ngroups = (a.R + 7) / 8;
    const uint32_t ktiles = ktiles_row / KS, kfirst = kh * ktiles;    // this set's k-steps
    const uint32_t klast = ktiles - 1;
    const uint32_t nx = (ntiles + WN * NT - 1) / (WN * NT), ny = (ngroups + 2 * GROUPS - 1) / (2 * GROUPS);
    uint32_t px, py;
    if (!xcd_tile(blockIdx.x, a.cols, nx, ny, px, py)) return;
    const uint32_t nt_wg = px * WN * NT, g_wg = py * 2 * GROUPS;
    const uint32_t lds0 = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)gemm_smem);

    // chunk c of a stage: weight tile nt_wg + c (c < WN * NT) or fragment group
    // g_wg + c - WN * NT; one past the end re-reads the last one, and its results are dropped
    // (GATED: of a wave's four tiles the first two are gates', the others their values')
    auto tile_of = [&](uint32_t v) {
        return GATED ? proj_paired_tile(v / 4 * 2 + v % 2, v / 2 % 2, ntiles) : min(v, ntiles - 1);
    };
    const unsigned char* src[CPW];
#pragma unroll
    for (int i = 0; i < CPW; i++) {
        const uint32_t c = wave * CPW + i;
        const unsigned char* p =
            c < WN * NT ? reinterpret_cast<const unsigned char*>(a.w) + (size_t)tile_of(nt_wg + c) * ktiles_row * 1024
                        : reinterpret_cast<const unsigned char*>(a.xfrag) +
                              (size_t)min(g_wg + c - WN * NT, ngroups - 1) * ktiles_row * 1024;
        src[i] = uniform_ptr(p + (size_t)kfirst * 1024);
    }
    const uint32_t lane_off = lane * 16;
    auto issue = [&](uint32_t kt) {                        // a k-step past the end copies the last one again
        const size_t k = (size_t)min(kt, klast) * 1024;
        const uint32_t to = lds0 + ((kt % RING) * KS + kh) * STAGE + wave * CPW * 1024;
#pragma unroll
        for (int i = 0; i < CPW; i++) lds_direct_load(to + i * 1024, src[i] + k, lane_off);
    };

    f32x4 acc[NT][GROUPS];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int gi = 0; gi < GROUPS; gi++) acc[t][gi] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
    for (int st0 = 0; st0 < RING - 1; st0++) issue(st0);
    const uint32_t w_off = wn * NT * 1024 + lane * 16;
    const uint32_t x_off = (WN * NT + wr * GROUPS) * 1024 + lane * 16;
    if constexpr (PIPE) {
        static_assert(RING >= 4, "a stage is read while the one before it is multiplied");
        half8 w0[NT], x0[GROUPS], w1[NT], x1[GROUPS];
        auto read_ops = [&](half8 (&wv)[NT], half8 (&xv)[GROUPS], uint32_t kt) {
            const unsigned char* st = gemm_smem + ((kt % RING) * KS + kh) * STAGE;
#pragma unroll
            for (int t = 0; t < NT; t++) wv[t] = *reinterpret_cast<const half8*>(st + w_off + t * 1024);
#pragma unroll
            for (int gi = 0; gi < GROUPS; gi++) xv[gi] = *reinterpret_cast<const half8*>(st + x_off + gi * 1024);
        };
        auto mfmas = [&](const half8 (&wv)[NT], const half8 (&xv)[GROUPS]) {
#pragma unroll
            for (int gi = 0; gi < GROUPS; gi++)
#pragma unroll
                for (int t = 0; t < NT; t++)
                    acc[t][gi] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv[t], xv[gi], acc[t][gi], 0, 0, 0);
        };
        // stage 0 into the first register set
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(CPW * (RING - 2)) : "memory");
        read_ops(w0, x0, 0);
        // Step kt: everybody's copies of stage kt + 1 have landed (the barrier),
        // the copies of stage kt + RING - 1 go to the slot of stage kt - 1, whose
        // last reads were waited for before the MFMAs of step kt - 1 were issued;
        // then the reads of stage kt + 1, then the MFMAs of stage kt.  Two steps
        // per iteration so that no register set is copied; a step past the end
        // reads a stage that holds a repeat of the last one and is not used.
        uint32_t kt = 0;
        // A step in quarters, a copy, then reads among the products: left alone, the compiler puts most reads behind the
        // products and waits for each few, and copies issued together keep a SIMD's two waves from the matrix pipe at
        // the same time.
        auto step = [&](const half8 (&wv)[NT], const half8 (&xv)[GROUPS], half8 (&wn_)[NT], half8 (&xn)[GROUPS], uint32_t k) {
            constexpr int PER = GROUPS / NT;
            static_assert(GROUPS % NT == 0 && CPW <= NT, "a quarter's share");
            const size_t from = (size_t)min(k + RING - 1, klast) * 1024;
            const uint32_t to = lds0 + ((k + RING - 1) % RING * KS + kh) * STAGE + wave * CPW * 1024;
            const unsigned char* st = gemm_smem + ((k + 1) % RING * KS + kh) * STAGE;
#pragma unroll
            for (int q = 0; q < NT; q++) {
                __builtin_amdgcn_sched_barrier(0);
                if (q < CPW) lds_direct_load(to + q * 1024, src[q] + from, lane_off);
                __builtin_amdgcn_sched_barrier(0);
                wn_[q] = *reinterpret_cast<const half8*>(st + w_off + q * 1024);
#pragma unroll
                for (int i = 0; i < PER; i++) xn[q * PER + i] = *reinterpret_cast<const half8*>(st + x_off + (q * PER + i) * 1024);
#pragma unroll
                for (int i = 0; i < PER; i++)
#pragma unroll
                    for (int t = 0; t < NT; t++)
                        acc[t][q * PER + i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv[t], xv[q * PER + i], acc[t][q * PER + i], 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 1 + PER; i++) {
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x008, NT * PER / (1 + PER), 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        constexpr bool PAIR = RING >= 5;                   // one barrier for two steps
        for (; kt + 2 <= ktiles; kt += 2) {
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (PAIR)
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(CPW * (RING - 4)) : "memory");
            else
                asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(CPW * (RING - 3)) : "memory");
            step(w0, x0, w1, x1, kt);
            if constexpr (!PAIR) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(CPW * (RING - 3)) : "memory");
            step(w1, x1, w0, x0, kt + 1);
        }
        if (kt < ktiles) mfmas(w0, x0);                   // odd number of k-steps
    } else
    for (uint32_t kt = 0; kt < ktiles; kt++) {
        // this wave's copies of stage kt have landed; those of the RING - 2 stages after it may be in flight
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(CPW * (RING - 2)) : "memory");
        issue(kt + RING - 1);
        const unsigned char* st = gemm_smem + ((kt % RING) * KS + kh) * STAGE;
        half8 wv[NT], xv[GROUPS];
#pragma unroll
        for (int t = 0; t < NT; t++) wv[t] = *reinterpret_cast<const half8*>(st + w_off + t * 1024);
#pragma unroll
        for (int gi = 0; gi < GROUPS; gi++) xv[gi] = *reinterpret_cast<const half8*>(st + x_off + gi * 1024);
#pragma unroll
        for (int gi = 0; gi < GROUPS; gi++)
#pragma unroll
            for (int t = 0; t < NT; t++)
                acc[t][gi] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv[t], xv[gi], acc[t][gi], 0, 0, 0);
        // all operand reads first (their latency overlaps, and the first MFMAs
        // hide the rest), then the MFMAs: left alone the scheduler reads two
        // fragments at a time and waits for each pair
        __builtin_amdgcn_sched_group_barrier(0x100, NT + GROUPS, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, NT * GROUPS, 0);
    }
    // the last steps' copies still target the ring
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    if constexpr (KS == 2) {
        // the upper half's sums through LDS (the rings are done with: every wave's
        // copies have landed and, past the barrier, every wave's reads are over),
        // added to the lower half's in a fixed order
        static_assert((size_t)WAVES * NT * GROUPS * 1024 <= (size_t)RING * KS * STAGE, "the partial tiles fit the rings");
        f32x4* red = reinterpret_cast<f32x4*>(gemm_smem) + (size_t)wave * NT * GROUPS * 64 + lane;
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (kh == 1) {
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int gi = 0; gi < GROUPS; gi++) red[(t * GROUPS + gi) * 64] = acc[t][gi];
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (kh == 1) return;
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int gi = 0; gi < GROUPS; gi++) {
                const f32x4 o = red[(t * GROUPS + gi) * 64];
#pragma unroll
                for (int i = 0; i < 4; i++) acc[t][gi][i] += o[i];
            }
    }

    const uint32_t nt0 = nt_wg + wn * NT, group0 = g_wg + wr * GROUPS;
    if (nt0 >= ntiles || group0 >= ngroups) return;
    if constexpr (GATED) {
#pragma unroll
        for (int t = 0; t < NT / 2; t++)
#pragma unroll
            for (int gi = 0; gi < GROUPS; gi++)
                proj_store_pair(a, acc[t][gi], acc[t + 2][gi], nt0 / 2 + t, group0 + gi, lane);
        return;
    }
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int gi = 0; gi < GROUPS; gi++) proj_store_tile(a, acc[t][gi], nt0 + t, group0 + gi, lane);
}

}  // namespace wr
