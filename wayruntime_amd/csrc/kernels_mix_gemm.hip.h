// Matrix products of mixer-stack models: bfloat16 weights in operand order,
// activation rows in fragment order (mix_common.hip.h), and the output put where
// the next step wants it: 32-bit or activation-type rows, or directly the
// fragment of the next product.
//
//   mix_gemm_split_kernel  any row count, both activation types: a workgroup's waves
//                          share a tile and split the input range (decode: HBM-bound
//                          on the weight bytes)
//   mix_gemm_runs_kernel   experts whose weights are large: HBM-bound on them up to some hundred rows each
//   mix_gemm_lds_kernel    prompt-sized row counts, bfloat16: 128-output tiles
//                          staged through LDS (MFMA-bound)
#pragma once

#include "mix_common.hip.h"

namespace wr {

constexpr uint32_t kMixOutRowsF32 = 0, kMixOutRows = 1, kMixOutFrag = 2, kMixOutSplit = 3, kMixOutGated = 4,
                   kMixOutSplitGated = 5;

struct MixGemmArgs {
    const bf16x8* w;
    const void* x;
    uint32_t ntiles, ktiles;         // of one matrix
    uint32_t x_kt, x_kt_z;
    uint32_t rows, groups;
    const int32_t* group_expert;
    uint32_t out, ldy, h_kt, col_z, n_split, silu_end, sigmoid_end, tanh_end, relu2, gelu;
    float scale, limit, slope, up_bias;
    const float* bias;
    uint32_t cols;                   // mix_gemm_lds_kernel without experts: XCDs that share out the outputs (xcd_tile);
                                     // a stream of experts: runs that the XCDs share out, or 0
    const uint32_t* x_perm;
    const float* x_scale;            // a factor per row of the input (applied to its products), or nullptr
    float* y;
    void* ya;
    void* h;
    float* part;                     // PARTS = 2: partial tiles [2][ntiles][64][4]
    uint32_t* tickets;               // ... one per tile, zero between launches
};

__global__ __launch_bounds__(256) void mix_pack_kernel(const uint16_t* __restrict__ w, u32x4* __restrict__ tiles,
                                                       uint64_t units, uint32_t K)
{
    const uint64_t unit = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (unit >= units) return;
    const uint32_t lane = (uint32_t)(unit & 63);
    const uint64_t tile = unit >> 6;
    const uint32_t kt = (uint32_t)(tile % (K / 32));
    const uint64_t nt = tile / (K / 32);
    tiles[unit] = *reinterpret_cast<const u32x4*>(w + ((nt * 16 + (lane & 15)) * K + kt * 32 + (lane >> 4) * 8));
}

template <bool F32>
__device__ __forceinline__ void mix_put4(void* p, size_t elem, f32x4 v)
{
    typename MixAct<F32>::V4 o;
#pragma unroll
    for (int i = 0; i < 4; i++) o[i] = (typename MixAct<F32>::E)v[i];
    *reinterpret_cast<typename MixAct<F32>::V4*>(reinterpret_cast<typename MixAct<F32>::E*>(p) + elem) = o;
}

// The gated unit of one gate and one up output.
template <bool F32>
__device__ __forceinline__ float mix_gated(const MixGemmArgs& a, float gate, float up)
{
    if (a.limit > 0.f) {                                   // (uniform, like gelu)
        gate = fminf(gate, a.limit);
        up = fminf(fmaxf(up, -a.limit), a.limit) + a.up_bias;
        return gate * mix_sigmoid<F32>(a.slope * gate) * up;
    }
    // the tanh form of GELU is x * logistic(2 y), y the argument of its tanh
    const float y = a.gelu ? 1.5957691216057308f * (gate + 0.044715f * gate * gate * gate) : gate;
    return gate * mix_sigmoid<F32>(y) * up;
}

// Bias and activation of outputs n .. n + 3.
template <bool F32>
__device__ __forceinline__ f32x4 mix_activate(const MixGemmArgs& a, f32x4 v, uint32_t n)
{
    if (a.bias) {
        const f32x4 b = *reinterpret_cast<const f32x4*>(a.bias + n);
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] += b[i];
    }
    if (n < a.sigmoid_end) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float s = mix_sigmoid<F32>(v[i]);
            v[i] = n + i < a.silu_end ? v[i] * s : (n + i < a.sigmoid_end ? s : v[i]);
        }
    } else if (n < a.tanh_end) {
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = n + i < a.tanh_end ? tanhf(v[i]) : v[i];
    } else if (a.relu2) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float p = fmaxf(v[i], 0.f);
            v[i] = p * p;
        }
    }
    return v;
}

// Accumulator tile nt of row group `group`: lane 16g + c holds outputs
// 16 nt + 4g .. +3 of row 16 group + c.  `up`: the tile's partner (GATED, SPLIT_GATED).
template <bool F32>
__device__ __forceinline__ void mix_store_tile(const MixGemmArgs& a, f32x4 v, f32x4 up, uint32_t nt, uint32_t group,
                                               uint32_t z, int lane)
{
    const uint32_t c = lane & 15, g = lane >> 4, row = group * 16 + c, n = nt * 16 + 4 * g;
    if (row >= a.rows || nt >= a.ntiles) return;
    if (a.x_scale) {
        const float s = a.x_scale[row];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            v[i] *= s;
            up[i] *= s;
        }
    }
    if (a.out >= kMixOutGated) {
        if (a.out == kMixOutSplitGated && nt * 16 < a.n_split) {
            *reinterpret_cast<f32x4*>(a.y + (size_t)row * a.ldy + n) = mix_activate<F32>(a, v, n);
            *reinterpret_cast<f32x4*>(a.y + (size_t)row * a.ldy + n + 16) = mix_activate<F32>(a, up, n + 16);
            return;
        }
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = mix_gated<F32>(a, v[i], up[i]);
        const uint32_t to = nt - (a.out == kMixOutSplitGated ? a.n_split / 16 : 0u);
        mix_put4<F32>(a.h, frag_elem(row, to / 2 * 16 + 4 * g, a.h_kt), v);
        return;
    }
    v = mix_activate<F32>(a, v, n);
    if (a.scale != 0.f) {
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] *= a.scale;
    }
    if (a.out == kMixOutRowsF32) {
        *reinterpret_cast<f32x4*>(a.y + (size_t)row * a.ldy + (size_t)z * a.col_z + n) = v;
    } else if (a.out == kMixOutRows) {
        mix_put4<F32>(a.ya, (size_t)row * a.ldy + n, v);
    } else if (a.out == kMixOutSplit && n >= a.n_split) {
        *reinterpret_cast<f32x4*>(a.y + (size_t)row * a.ldy + n - a.n_split) = v;
    } else {
        mix_put4<F32>(a.h, frag_elem(row, z * a.col_z + n, a.h_kt), v);
    }
}

// A workgroup's WAVES waves share NT x 16 outputs and GR x 16 rows and take an equal
// part of the input range each; their sums meet in LDS and are added in wave order,
// every wave adding and storing its share of the tiles.  A wave keeps D k-steps on
// their way (operands from HBM are one to three microseconds away under load):
// loads stand behind the products that free their registers; in whole turns of D
// none is conditional, so the compiler's count of loads in flight is exact, and what
// is left behind the last turn is asked for all at once (in registers of its own name:
// kept in those of the turns, the compiler holds both).  One after the other they were a
// trip to memory each: 16 rows, 768 -> 2048 5.5 us, 3.9 now; 1536 -> 512 5.5, 4.3.
// Few rows: bound by the weights' bytes.  More rows: by the bytes that pass a
// compute unit's vector cache, NT + GR KiB a k-step for NT x GR products.
// STREAM: every weight tile is read by one workgroup only (no use in keeping it).
// With group_expert the GR groups share an expert (GR divides tile_groups), and of a run's only those are read,
// multiplied and stored that rows are in: a compute unit takes in 47 KiB a microsecond, 2 of weights and one for each
// group of rows with every k-step.  64 experts, 48 rows each give or take a third, 2048 -> 1024: groups of four with the
// empty ones 68 us, without them 64, all eight that a run may have in one workgroup 62, its workgroups on one XCD
// 58; 64 rows each 88 (LDS tiles) -> 64.  PICKED: the same of single groups (tile_groups 1) in any order, cut at every
// GR-th; alone a group has twice the k-steps on their way.
//
// PARTS = 2 (one group of rows, one matrix, no gate): two workgroups take half of the
// input range each, and the one that draws the tile's second ticket adds the other's
// partial tile (a sum of two: the same bits either way).  A narrow weight has 128 tiles
// for 256 compute units, and a unit takes in 46 GB/s of weights and rows at best, so
// half of them idle is half the rate.  16 rows, weights from HBM: 8192 -> 2048 11.5 -> 9.4
// us, -> 512 10.6 -> 7.8; 6144 -> 2048 9.4 -> 7.8; 4096 -> 2048 7.0 -> 6.6, -> 1024 6.7 ->
// 6.0; at 2048 inputs the exchange costs more (4.8 -> 5.2).
// SETS: so many sets of WAVES waves, each with tiles of its own.  (The arguments by value: by reference the loads come out in another order, 1 to
// 4 % slower for one tile over inputs that are no power of two.)
template <bool F32, int NT, int GR, int WAVES, int DEPTH, bool STREAM, int PARTS, bool PICKED, int SETS = 1>
__device__ __forceinline__ void mix_gemm_split(const MixGemmArgs a, uint32_t bx, uint32_t by, uint32_t z)
{
    using V8 = typename MixAct<F32>::V8;
    constexpr uint32_t SET = WAVES * NT * GR * 64;
    __shared__ f32x4 s_part[SETS * SET];
    const int lane = threadIdx.x & 63;
    uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t mine = SETS > 1 ? wave / WAVES * SET : 0;
    if constexpr (SETS > 1) {
        bx = bx * SETS + wave / WAVES;
        wave %= WAVES;
    }
    static_assert(PARTS == 1 || (PARTS == 2 && NT == 1 && GR == 1), "one tile, two halves");
    if constexpr (STREAM && GR > 1 && !PICKED) {
        if (a.cols) {                                      // runs, up to a multiple of 8: a run's workgroups on one XCD
            const uint32_t id = by * gridDim.x + bx, in_xcd = id / 8, y = in_xcd / gridDim.x * 8 + id % 8;
            bx = in_xcd % gridDim.x;
            by = y < a.cols ? y * (8 / GR) : (y - a.cols) * (8 / GR) + 1;       // GR = 4: first halves of all runs, then the second
            if (by * GR >= a.groups) return;
        }
    }
    const uint32_t nt0 = bx * NT, group0 = PARTS > 1 ? 0 : PICKED ? by : by * GR, part = PARTS > 1 ? by : 0;
    uint32_t mat = z, live = GR;                           // live: groups that rows are in (those of a run come first)
    if (a.group_expert) {
        const int e = a.group_expert[group0];
        if (e < 0) return;                                 // uniform over the workgroup
        mat = (uint32_t)e;
        if constexpr (PICKED) {                            // single groups: those of an expert that stand together, GR at most
            if (group0 % GR && a.group_expert[group0 - 1] == e) return;
            live = 1;
            for (uint32_t i = group0 + 1; i % GR && i < a.groups && a.group_expert[i] == e; i++) live++;
        } else if constexpr (STREAM && GR > 1) {
            live = 1;
#pragma unroll
            for (uint32_t i = 1; i < GR; i++)
                if (a.group_expert[group0 + i] >= 0) live = i + 1;
        }
    }
    const uint32_t k_begin = a.ktiles * (part * WAVES + wave) / (PARTS * WAVES),
                   n = a.ktiles * (part * WAVES + wave + 1) / (PARTS * WAVES) - k_begin;

    const bf16x8* wp[NT];
    const V8* xp[GR];
#pragma unroll
    for (int t = 0; t < NT; t++)
        wp[t] = a.w + (((size_t)mat * a.ntiles + min(nt0 + t, a.ntiles - 1)) * a.ktiles + k_begin) * 64;
#pragma unroll
    for (int i = 0; i < GR; i++)
        xp[i] = reinterpret_cast<const V8*>(a.x) + ((size_t)min(group0 + i, a.groups - 1) * a.x_kt + (size_t)z * a.x_kt_z + k_begin) * 64;
    uint32_t x_lane[GR];
#pragma unroll
    for (int i = 0; i < GR; i++) x_lane[i] = lane;
    if constexpr (GR == 1 || PICKED) {
        if (a.x_perm) {                                    // rows picked one by one: the operand's lanes fetch their own
#pragma unroll
            for (int i = 0; i < GR; i++) {
                const uint32_t pick = a.x_perm[min(group0 + i, a.groups - 1) * 16 + (lane & 15)], row = pick == 0xFFFFFFFFu ? 0 : pick;
                xp[i] = reinterpret_cast<const V8*>(a.x) + (size_t)k_begin * 64;
                x_lane[i] = (row >> 4) * a.x_kt * 64 + (lane & 48) + (row & 15);
            }
        }
    }

    const auto product = [&](auto groups) {
        constexpr int L = decltype(groups)::value, D = PICKED && L == 1 ? 2 * DEPTH : DEPTH;
        f32x4 acc[NT][L];
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int i = 0; i < L; i++) acc[t][i] = f32x4{0.f, 0.f, 0.f, 0.f};

        bf16x8 w[D][NT];
        V8 x[D][L];
        auto load = [&](bf16x8 (&wv)[NT], V8 (&xv)[L], uint32_t k) {
#pragma unroll
            for (int t = 0; t < NT; t++)
                wv[t] = STREAM ? __builtin_nontemporal_load(&wp[t][k * 64 + lane]) : wp[t][k * 64 + lane];
#pragma unroll
            for (int i = 0; i < L; i++) xv[i] = xp[i][k * 64 + x_lane[i]];
        };
        auto multiply = [&](const bf16x8 (&wv)[NT], const V8 (&xv)[L]) {
#pragma unroll
            for (int i = 0; i < L; i++)
#pragma unroll
                for (int t = 0; t < NT; t++) acc[t][i] = mix_mfma(wv[t], xv[i], acc[t][i]);
        };
        if constexpr (F32) {
            // Half a turn is asked for, then the other half multiplied: eight 32-bit products to a tile and k-step are as long
            // as a load, and asked for behind them it is late (4096 -> 4096 at 24 rows 26.2 us, 21.2 now; gated, one row,
            // 1536 -> 4096 9.8, 8.3).  Past the end the last step is read again and not used.
            constexpr int H = D / 2;
            auto ask = [&](int d, uint32_t k) {
#pragma unroll
                for (int u = 0; u < H; u++) load(w[d + u], x[d + u], min(k + u, n - 1));
            };
            auto take = [&](int d, uint32_t k) {
#pragma unroll
                for (int u = 0; u < H; u++)
                    if (k + u < n) multiply(w[d + u], x[d + u]);
            };
            if (n) ask(0, 0);
            for (uint32_t k = 0; k < n; k += D) {
                ask(H, k + H);
                take(0, k);
                ask(0, k + D);
                take(H, k + H);
            }
        }
        const uint32_t turns = F32 ? 0 : n / D, rest = F32 ? 0 : n - turns * D;
        if (turns) {
#pragma unroll
            for (int d = 0; d < D; d++) load(w[d], x[d], d);
            for (uint32_t turn = 1; turn < turns; turn++) {
#pragma unroll
                for (int d = 0; d < D; d++) {
                    multiply(w[d], x[d]);
                    load(w[d], x[d], turn * D + d);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
#pragma unroll
            for (int d = 0; d < D; d++) multiply(w[d], x[d]);
        }
        if (__builtin_expect(rest != 0, 0)) {
            bf16x8 wr[D - 1][NT];
            V8 xr[D - 1][L];
#pragma unroll
            for (int d = 0; d < D - 1; d++)
                if ((uint32_t)d < rest) load(wr[d], xr[d], turns * D + d);
#pragma unroll
            for (int d = 0; d < D - 1; d++)
                if ((uint32_t)d < rest) multiply(wr[d], xr[d]);
        }

#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int i = 0; i < L; i++) s_part[mine + ((wave * NT + t) * GR + i) * 64 + lane] = acc[t][i];
    };
    if constexpr (STREAM && GR > 1) {
        static_assert(GR == 4 || GR == 8);
        switch (live) {
        case 1: product(std::integral_constant<int, 1>()); break;
        case 2: product(std::integral_constant<int, 2>()); break;
        case 3: product(std::integral_constant<int, 3>()); break;
        case 4: product(std::integral_constant<int, 4>()); break;
        default:
            if constexpr (GR == 8) {
                switch (live) {
                case 5: product(std::integral_constant<int, 5>()); break;
                case 6: product(std::integral_constant<int, 6>()); break;
                case 7: product(std::integral_constant<int, 7>()); break;
                default: product(std::integral_constant<int, 8>()); break;
                }
            }
        }
    } else {
        product(std::integral_constant<int, GR>());
    }
    lds_barrier();
    auto sum = [&](uint32_t i) {
        f32x4 v = s_part[mine + i * 64 + lane];
#pragma unroll
        for (int p = 1; p < WAVES; p++) {
            const f32x4 o = s_part[mine + (p * NT * GR + i) * 64 + lane];
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] += o[j];
        }
        return v;
    };
    if constexpr (PARTS > 1) {
        if (wave > 0) return;
        f32x4 v = sum(0);
        float* mine = a.part + ((size_t)(part * a.ntiles + nt0) * 64 + lane) * 4;
#pragma unroll
        for (int j = 0; j < 4; j++) part_store(mine + j, v[j]);
        // the stores are acknowledged before the ticket is drawn: who draws the second one reads them
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        uint32_t ticket = 0;
        if (lane == 0) ticket = __hip_atomic_fetch_add(&a.tickets[nt0], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__builtin_amdgcn_readfirstlane(ticket) == 0) return;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        const float* other = a.part + ((size_t)((1 - part) * a.ntiles + nt0) * 64 + lane) * 4;
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] += part_load(other + j);
        if (lane == 0) a.tickets[nt0] = 0;
        mix_store_tile<F32>(a, v, v, nt0, 0, z, lane);
        return;
    }
    if (a.out >= kMixOutGated) {
        if constexpr (NT % 2 == 0) {
#pragma unroll 1
            for (uint32_t u = wave; u < NT / 2 * GR; u += WAVES) {
                const uint32_t t = u / GR * 2, i = u % GR;
                if (i >= live) continue;
                mix_store_tile<F32>(a, sum(t * GR + i), sum((t + 1) * GR + i), nt0 + t, group0 + i, z, lane);
            }
        }
        return;
    }
#pragma unroll 1
    for (uint32_t u = wave; u < NT * GR; u += WAVES) {
        if (u % GR >= live) continue;
        const f32x4 v = sum(u);
        mix_store_tile<F32>(a, v, v, nt0 + u / GR, group0 + u % GR, z, lane);
    }
}

// REGION: an XCD's workgroups take neighbouring tiles (xcd_region).  A form of its own: asked in the kernel, the question was 0.2 us of every launch.
template <bool F32, int NT, int GR, int WAVES, int DEPTH, bool STREAM, int PARTS = 1, bool PICKED = false, bool REGION = false>
__global__ __launch_bounds__(WAVES * 64, WAVES > 4 ? 1 : 2) void mix_gemm_split_kernel(const MixGemmArgs a)
{
    const uint32_t bx = REGION ? xcd_region(blockIdx.x, (a.ntiles + NT - 1) / NT) : blockIdx.x;
    mix_gemm_split<F32, NT, GR, WAVES, DEPTH, STREAM, PARTS, PICKED>(a, bx, blockIdx.y, blockIdx.z);
}

// Two products of up to sixteen rows that do not wait for each other: a's batch of matrices, and a small one whose few tiles took a launch
// of their own (16 rows, four of 2048 -> 2048 and 2048 -> 64: 8.7 and 4.6 us, 10.6 together).  Each in the form that it has alone, so the
// same bits: four waves to a tile of the small one's, a workgroup's other four with the next.
// The small one's workgroups come first: they end as the others do.
template <int WAVES, int DEPTH, bool REGION>
__global__ __launch_bounds__(WAVES * 64, WAVES > 4 ? 1 : 2) void mix_gemm_two_kernel(const MixGemmArgs a, const MixGemmArgs b)
{
    constexpr int SETS = WAVES / 4;
    const uint32_t of_b = (b.ntiles + SETS - 1) / SETS, of_a = (a.ntiles + 1) / 2;
    const uint32_t item = REGION ? xcd_region(blockIdx.x, gridDim.x) : blockIdx.x;
    if (item < of_b) {
        mix_gemm_split<false, 1, 1, 4, 8, true, 1, false, SETS>(b, item, 0, 0);
    } else {
        const uint32_t i = item - of_b;
        mix_gemm_split<false, 2, 1, WAVES, DEPTH, true, 1, false>(a, i % of_a, 0, i / of_a);
    }
}

// Products of experts whose weights are large, as a stream of them.  A piece of work is up to eight groups of rows that
// share an expert (a run's; SINGLE: an expert's that stand together) against WAVES x NT tiles of its outputs: a wave has
// NT tiles over the whole input range, weights straight to registers (each byte is one wave's), two chunks of KC
// k-steps on their way; the rows pass through LDS, a chunk in two buffers, for all waves.
// Bound by HBM.  mix_gemm_split_kernel, which splits the input range over its waves, reads the rows once for every two tiles
// (1.5 times the weights' bytes at 48 rows an expert), this one once for eight, and a piece's workgroups are on one XCD,
// whichever runs there are (dealt out to all of them: 51 us -> 70).  Us, split kernel / this one: 64 experts, 2048 ->
// 1024 in runs of 48 rows each 62.5 / 52 (5.2 TB/s; 20: 49 / 47, 128: 108, tiles, / 92), 4096 -> 4096 of 32 at 48
// 235 / 186 (5.8 TB/s), 4096 -> 14 336 of 8 at 60 223 / 174; single groups, 64 experts of 2048 -> 1024 with 29 rows each 68 /
// 48, picked one by one 76 / 53, 4096 -> 384 85 / 39.
// Tried: two chunks of rows on their way (51.7 -> 54.5), four tiles to a wave (60 -> 65), one (60 -> 58.6 but 1024 -> 2048
// 62 -> 65), two waves (62); a loop over pieces around this (spills, 52 -> 60).
// What pieces are cut from, at most: a wave finds them with a ballot for every 64.
constexpr uint32_t kMixStreamRuns = 256, kMixStreamGroups = 512;       // (groups: SINGLE)

// The launch's arguments, read again: what a kernel's end needs of them is not kept through its loops.
__device__ __forceinline__ const MixGemmArgs& mix_fresh_args()
{
    typedef const __attribute__((address_space(4))) MixGemmArgs* Args;
    Args p = (Args)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const MixGemmArgs*)p;
}

// One wave: tiles nt0 .. nt0 + tiles - 1 of the groups first, first + step, ..., one after the other: for orders of groups that
// nobody makes in earnest (routing puts an expert's together), so that they are right all the same.
__device__ __forceinline__ void mix_gemm_scattered(const MixGemmArgs& a, uint32_t nt0, uint32_t tiles, uint32_t first, uint32_t step, int lane)
{
    if (nt0 >= a.ntiles) return;
    for (uint32_t group = first; group < a.groups; group += step) {
        const int e = a.group_expert[group];
        if (e < 0) continue;
        const bf16x8* x = reinterpret_cast<const bf16x8*>(a.x) + (size_t)group * a.x_kt * 64 + lane;
        if (a.x_perm) {
            const uint32_t pick = a.x_perm[group * 16 + (lane & 15)], row = pick == 0xFFFFFFFFu ? 0 : pick;
            x = reinterpret_cast<const bf16x8*>(a.x) + (size_t)(row >> 4) * a.x_kt * 64 + (lane & 48) + (row & 15);
        }
#pragma unroll 1
        for (uint32_t t = 0; t < tiles; t += 2) {
            const uint32_t nt = nt0 + t;
            const bf16x8* w0 = a.w + ((size_t)(uint32_t)e * a.ntiles + min(nt, a.ntiles - 1)) * a.ktiles * 64 + lane;
            const bf16x8* w1 = a.w + ((size_t)(uint32_t)e * a.ntiles + min(nt + 1, a.ntiles - 1)) * a.ktiles * 64 + lane;
            f32x4 v0 = f32x4{0.f, 0.f, 0.f, 0.f}, v1 = v0;
            for (uint32_t k = 0; k < a.ktiles; k++) {
                const bf16x8 xv = x[k * 64];
                v0 = mix_mfma(w0[k * 64], xv, v0);
                v1 = mix_mfma(w1[k * 64], xv, v1);
            }
            mix_store_tile<false>(a, v0, v1, nt, group, 0, lane);
            if (a.out < kMixOutGated) mix_store_tile<false>(a, v1, v1, nt + 1, group, 0, lane);
        }
    }
}

template <int NT, int WAVES, int KC, bool SINGLE>
__global__ __launch_bounds__(WAVES * 64, 2) void mix_gemm_runs_kernel(const MixGemmArgs a)
{
    constexpr uint32_t MOST = SINGLE ? kMixStreamGroups : kMixStreamRuns;
    static_assert(MOST % 64 == 0);
    constexpr int GR = 8, D = 2 * KC, WORDS = MOST / 64, RUN = SINGLE ? 1 : GR;
    __shared__ bf16x8 s_x[2][KC * GR * 64];
    const int lane = threadIdx.x & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t n = a.ktiles, last = n - 1;
    // Where pieces begin, a bit to a run or group.
    const uint32_t entries = a.groups / RUN, units = (a.ntiles + NT * WAVES - 1) / (NT * WAVES);
    uint64_t begins[WORDS], edges[WORDS];                  // edges (SINGLE): where an expert's groups end or begin
    int expert_of[WORDS];
#pragma unroll
    for (int i = 0; i < WORDS; i++) {
        const uint32_t at = i * 64 + lane;
        expert_of[i] = -1;
        if (at < entries) expert_of[i] = a.group_expert[at * RUN];
    }
    uint32_t pieces = 0, start = 0;
    int before = -1;
#pragma unroll
    for (int i = 0; i < WORDS; i++) {
        const int e = expert_of[i];
        bool begin = e >= 0;
        if constexpr (SINGLE) {                            // the first of an expert's groups, and every eighth behind it
            int prev = __shfl_up(e, 1, 64);
            if (lane == 0) prev = before;
            edges[i] = __ballot(e < 0 || e != prev);
            const uint64_t firsts = __ballot(e >= 0 && e != prev), upto = firsts & (~0ull >> (63 - lane));
            const uint32_t first = upto ? i * 64 + 63 - __builtin_clzll(upto) : start;
            begin = begin && (i * 64 + lane - first) % GR == 0;
            if (firsts) start = i * 64 + 63 - __builtin_clzll(firsts);
            before = __builtin_amdgcn_readlane(e, 63);
        }
        begins[i] = __ballot(begin);
        pieces += (uint32_t)__popcll(begins[i]);
    }
    const uint32_t xcd = blockIdx.x % 8, work = pieces * units;
    if constexpr (SINGLE) {
        if (work > gridDim.x) {                            // an expert's groups all over the place: more pieces than there are workgroups
            const uint32_t step = gridDim.x / units, first = blockIdx.x / units;
            if (first < step) mix_gemm_scattered(a, (blockIdx.x % units * WAVES + wave) * NT, NT, first, step, lane);
            return;
        }
    }
    // XCD x takes an eighth of the pieces, one after the other: a run's rows come into one L2
    const uint32_t j = (uint32_t)((uint64_t)work * xcd / 8) + blockIdx.x / 8;
    if (j >= (uint32_t)((uint64_t)work * (xcd + 1) / 8)) return;
    uint32_t skip = j / units, group0 = 0, expert = 0, live = GR;        // live: groups that rows are in (they come first)
    bool found = false;
#pragma unroll
    for (int i = 0; i < WORDS; i++) {
        const uint32_t here = (uint32_t)__popcll(begins[i]);
        if (!found && skip < here) {
            uint64_t m = begins[i];
            for (uint32_t s = 0; s < skip; s++) m &= m - 1;
            const uint32_t bit = (uint32_t)__builtin_ctzll(m);
            const int e = __builtin_amdgcn_readlane(expert_of[i], (int)bit);
            group0 = (i * 64 + bit) * RUN;
            if constexpr (SINGLE) {
                const uint64_t behind = (edges[i] >> bit) >> 1 | (i + 1 < WORDS && bit ? edges[i + 1 < WORDS ? i + 1 : i] << (63 - bit) : 0);
                expert = (uint32_t)e;
                live = behind ? min((uint32_t)__builtin_ctzll(behind) + 1, (uint32_t)GR) : GR;
                live = min(live, a.groups - group0);
            } else {
                expert = (uint32_t)e;
                live = 1;
#pragma unroll
                for (uint32_t g = 1; g < GR; g++)
                    if (a.group_expert[group0 + g] >= 0) live = g + 1;
            }
            found = true;
        }
        if (!found) skip -= here;
    }
    const uint32_t nt0 = (j % units * WAVES + wave) * NT;

    const bf16x8* wp[NT];
#pragma unroll
    for (int t = 0; t < NT; t++)
        wp[t] = a.w + ((size_t)expert * a.ntiles + min(nt0 + t, a.ntiles - 1)) * n * 64;

    const auto product = [&](auto groups) {
        constexpr int L = decltype(groups)::value, S = (KC * L + WAVES - 1) / WAVES;
        f32x4 acc[NT][L];
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int i = 0; i < L; i++) acc[t][i] = f32x4{0.f, 0.f, 0.f, 0.f};
        bf16x8 w[D][NT], xr[S];
        // a wave's share of a chunk: blocks of one group and k-step
        const bf16x8* xp[S];
        uint32_t x_lane[S];
#pragma unroll
        for (int s = 0; s < S; s++) {
            const uint32_t b = min(wave + s * WAVES, (uint32_t)(KC * L - 1)), group = group0 + b / KC;
            xp[s] = reinterpret_cast<const bf16x8*>(a.x) + (size_t)group * a.x_kt * 64;
            x_lane[s] = lane;
            if constexpr (SINGLE) {
                if (a.x_perm) {                        // rows picked one by one: the lanes fetch their own
                    const uint32_t pick = a.x_perm[group * 16 + (lane & 15)], row = pick == 0xFFFFFFFFu ? 0 : pick;
                    xp[s] = reinterpret_cast<const bf16x8*>(a.x);
                    x_lane[s] = (row >> 4) * a.x_kt * 64 + (lane & 48) + (row & 15);
                }
            }
        }
        auto ask_rows = [&](uint32_t k0) {
#pragma unroll
            for (int s = 0; s < S; s++) {
                const uint32_t b = min(wave + s * WAVES, (uint32_t)(KC * L - 1));
                xr[s] = xp[s][min(k0 + b % KC, last) * 64 + x_lane[s]];
            }
        };
        auto put_rows = [&](int buf) {
#pragma unroll
            for (int s = 0; s < S; s++) {
                const uint32_t b = min(wave + s * WAVES, (uint32_t)(KC * L - 1));
                s_x[buf][(b % KC * L + b / KC) * 64 + lane] = xr[s];
            }
        };
        auto ask_weights = [&](int d, uint32_t k) {
#pragma unroll
            for (int t = 0; t < NT; t++) w[d][t] = __builtin_nontemporal_load(&wp[t][min(k, last) * 64 + lane]);
        };
        auto multiply = [&](int d) {
            bf16x8 xv[L];
#pragma unroll
            for (int i = 0; i < L; i++) xv[i] = s_x[d / KC][(d % KC * L + i) * 64 + lane];
#pragma unroll
            for (int i = 0; i < L; i++)
#pragma unroll
                for (int t = 0; t < NT; t++) acc[t][i] = mix_mfma(w[d][t], xv[i], acc[t][i]);
        };
        ask_rows(0);
#pragma unroll
        for (int d = 0; d < D; d++) ask_weights(d, d);
        put_rows(0);
        lds_barrier();
        uint32_t k = 0;
        for (; k + D < n; k += D) {
#pragma unroll
            for (int d = 0; d < D; d++) {
                if (d % KC == 0) ask_rows(k + d + KC);
                multiply(d);
                ask_weights(d, k + D + d);
                __builtin_amdgcn_sched_barrier(0);
                if (d % KC == KC - 1) {
                    put_rows(1 - d / KC);
                    lds_barrier();
                }
            }
        }
        ask_rows(k + KC);
#pragma unroll
        for (int d = 0; d < D; d++) {
            if (k + d < n) multiply(d);
            if (d == KC - 1) {
                put_rows(1);
                lds_barrier();
            }
        }
        const MixGemmArgs& o = mix_fresh_args();
        if (o.out >= kMixOutGated) {
            if constexpr (NT % 2 == 0)
#pragma unroll
                for (int t = 0; t < NT; t += 2)
#pragma unroll
                    for (int i = 0; i < L; i++) mix_store_tile<false>(o, acc[t][i], acc[t + 1][i], nt0 + t, group0 + i, 0, lane);
            return;
        }
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int i = 0; i < L; i++) mix_store_tile<false>(o, acc[t][i], acc[t][i], nt0 + t, group0 + i, 0, lane);
    };
    switch (live) {
    case 1: product(std::integral_constant<int, 1>()); break;
    case 2: product(std::integral_constant<int, 2>()); break;
    case 3: product(std::integral_constant<int, 3>()); break;
    case 4: product(std::integral_constant<int, 4>()); break;
    case 5: product(std::integral_constant<int, 5>()); break;
    case 6: product(std::integral_constant<int, 6>()); break;
    case 7: product(std::integral_constant<int, 7>()); break;
    default: product(std::integral_constant<int, 8>()); break;
    }
}

// Whether XCDs take whole matrices of a batch, one after the other, so that a matrix's weights and rows come into one L2 and no other;
// fewer than sixteen, and numbers that eight does not divide, are shared out tile by tile (us, so / every XCD for every matrix: 2047
// rows, 32 of 512 -> 128 19.6 / 23.6, 16 of 1024 -> 512 42.5 / 44.2, 700 rows 23.4 / 28.1; against 8 of 1024 -> 2048 into 32-bit rows at 2047
// 81.3 / 74.6, at 511 less by 9 %; two and four, on four and two XCDs each, 0.99 to 1.02 of the time on average and up to 1.12).
__host__ __device__ __forceinline__ bool mix_batch_apart(uint32_t batch) { return batch >= 16 && batch % 8 == 0; }

// 2 x 2 waves of 64 outputs x 16 GROUPS rows each: 128 outputs x 32 GROUPS rows a
// workgroup.  Per k-step 8 weight tiles and 2 GROUPS fragments, one KiB each and
// already in operand order, go to LDS by direct loads two k-steps ahead in a ring
// of three stages; lane i reads its operands back at 16 i.  With group_expert a
// workgroup's row groups share one expert.
//
// KS = 2: two such sets of waves, a ring of four stages each, take one half of the
// input range each (an even number of k-steps), and read a k-step's operands while the
// one before it is multiplied; the upper half's sums pass through LDS and are added to
// the lower half's.  For launches of one workgroup per compute unit and a long input
// range: twice the waves per SIMD, half the chain.
// 2047 rows, 8192 -> 2048, GROUPS 4: 93 -> 73 us, by quarters 68; 1000 rows, GROUPS 2: 80 -> 55.  (One barrier for two steps is
// up to 3 % faster there, and 10 to 17 % slower where weights come from HBM: 700 rows, 12 288 -> 4096 94 / 110.)
//
// WN = 4: eight waves, 256 outputs, a ring of five stages (160 KiB) and a barrier for two k-steps; a step goes by quarters (as
// with KS = 2 and GROUPS 4), a copy, then reads of the next step's operands among the products.  Bound by the matrix pipes at the clock the device grants them:
// a full device's step of 256 x 256 x 32 is 0.78 us, 0.51 of it products at 2.05 GHz, on 64 units alone 0.56 (2.4 GHz).  4095 rows,
// 8192 -> 4096 216 -> 194 us (1.42 PFLOP/s).  On the way there: operands read behind the barrier and a barrier a step 0.83, read a step ahead
// 0.80, the copies among the products 0.78.
template <int GROUPS, int KS = 1, int WN = 2>
constexpr int mix_gemm_ring() { return WN == 4 || (KS == 2 && GROUPS == 4) ? 5 : KS == 2 ? 4 : 3; }
template <int GROUPS, int KS = 1, int WN = 2>
constexpr size_t mix_gemm_lds_bytes() { return (size_t)KS * mix_gemm_ring<GROUPS, KS, WN>() * (4 * WN + 2 * GROUPS) * 1024; }

// BATCH: matrices of a batch (without it the kernel is that of one matrix alone: the share-out's code ahead of each
// workgroup's first load cost 2 to 3 %, 2047 rows, 2048 -> 14 400 gated 113.8 -> 117.5 us).
template <int GROUPS, int KS = 1, int WN = 2, bool BATCH = false>
__global__ __launch_bounds__(128 * WN * KS, KS == 2 || WN == 4 ? 1 : 2) void mix_gemm_lds_kernel(const MixGemmArgs a)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char mix_smem[];
    constexpr int NT = 4, WAVES = 2 * WN, TILES = WN * NT, CHUNKS = TILES + 2 * GROUPS, CPW = CHUNKS / WAVES, RING = mix_gemm_ring<GROUPS, KS, WN>();
    static_assert(CHUNKS % WAVES == 0, "every wave copies the same number of chunks");
    static_assert(WN == 2 || KS == 1);
    constexpr uint32_t STAGE = CHUNKS * 1024;
    const int lane = threadIdx.x & 63;
    const uint32_t wave_wg = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t kh = wave_wg / WAVES, wave = wave_wg % WAVES;   // half of the input range, wave of the set
    const uint32_t wn = wave % WN, wr = wave / WN;
    const uint32_t ktiles = a.ktiles / KS;                 // this set's k-steps
    const uint32_t nx = (a.ntiles + TILES - 1) / TILES, ny = (a.groups + 2 * GROUPS - 1) / (2 * GROUPS);
    uint32_t px, py, z = 0;
    if constexpr (BATCH) {
        z = blockIdx.y;
        if (mix_batch_apart(gridDim.y)) {
            const uint32_t id = blockIdx.y * gridDim.x + blockIdx.x, slot = id / 8, at = slot % gridDim.x;
            z = slot / gridDim.x * 8 + id % 8;
            px = at / ny;
            py = at % ny;
        } else if (!xcd_tile(blockIdx.x, a.cols, nx, ny, px, py)) {
            return;
        }
    } else if (!a.group_expert) {
        if (!xcd_tile(blockIdx.x, a.cols, nx, ny, px, py)) return;
    } else {
        // XCD x takes the output panels x, x + 8, ...: up to four side by side through all row panels, so that the rows
        // (few per expert, and each expert has weights of its own) are fetched into the XCD's L2 once for the four
        const uint32_t xcd = blockIdx.x % 8, slot = blockIdx.x / 8, share = (nx + 7) / 8;
        const uint32_t side = share % 4 == 0 ? 4u : (share % 2 == 0 ? 2u : 1u);
        // (fewer panels than XCDs: panels and rows dealt out as they come, or most XCDs would stand idle)
        const bool few = nx < 8;
        px = few ? blockIdx.x % nx : (slot / (ny * side) * side + slot % side) * 8 + xcd;
        py = few ? blockIdx.x / nx : slot / side % ny;
        if (px >= nx) return;
    }
    const uint32_t nt_wg = px * TILES, g_wg = py * 2 * GROUPS;
    uint32_t mat = z;
    if (a.group_expert) {
        const int e = a.group_expert[g_wg];
        if (e < 0) return;
        mat = (uint32_t)e;
    }
    const uint32_t klast = ktiles - 1;
    const uint32_t lds0 = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)mix_smem);
    const unsigned char* src[CPW];
#pragma unroll
    for (int i = 0; i < CPW; i++) {
        const uint32_t c = wave * CPW + i;
        const unsigned char* p =
            c < TILES ? reinterpret_cast<const unsigned char*>(a.w) +
                        ((size_t)mat * a.ntiles + min(nt_wg + c, a.ntiles - 1)) * a.ktiles * 1024
                  : reinterpret_cast<const unsigned char*>(a.x) +
                        ((size_t)min(g_wg + c - TILES, a.groups - 1) * a.x_kt + (size_t)z * a.x_kt_z) * 1024;
        src[i] = uniform_ptr(p + (size_t)kh * ktiles * 1024);
    }
    const uint32_t lane_off = lane * 16;
    auto issue = [&](uint32_t kt) {
        const size_t k = (size_t)min(kt, klast) * 1024;
        const uint32_t to = lds0 + ((kt % RING) * KS + kh) * STAGE + wave * CPW * 1024;
#pragma unroll
        for (int i = 0; i < CPW; i++) lds_direct_load(to + i * 1024, src[i] + k, lane_off);
    };

    f32x4 acc[NT][GROUPS];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int i = 0; i < GROUPS; i++) acc[t][i] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
    for (int st0 = 0; st0 < RING - 1; st0++) issue(st0);
    const uint32_t w_off = wn * NT * 1024 + lane * 16, x_off = (TILES + wr * GROUPS) * 1024 + lane * 16;
    auto read_ops = [&](bf16x8 (&wv)[NT], bf16x8 (&xv)[GROUPS], uint32_t kt) {
        const unsigned char* st = mix_smem + ((kt % RING) * KS + kh) * STAGE;
#pragma unroll
        for (int t = 0; t < NT; t++) wv[t] = *reinterpret_cast<const bf16x8*>(st + w_off + t * 1024);
#pragma unroll
        for (int i = 0; i < GROUPS; i++) xv[i] = *reinterpret_cast<const bf16x8*>(st + x_off + i * 1024);
    };
    auto multiply = [&](const bf16x8 (&wv)[NT], const bf16x8 (&xv)[GROUPS]) {
#pragma unroll
        for (int i = 0; i < GROUPS; i++)
#pragma unroll
            for (int t = 0; t < NT; t++) acc[t][i] = mix_mfma(wv[t], xv[i], acc[t][i]);
    };
    if constexpr (RING == 5) {
        bf16x8 w0[NT], x0[GROUPS], w1[NT], x1[GROUPS];
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(CPW * (RING - 2)) : "memory");
        read_ops(w0, x0, 0);
        // PAIR, two steps to a barrier: stages kt + 1 and kt + 2 have landed, kt + 3 may be in flight, kt + 4 and kt + 5 go where
        // kt - 1 and kt were, whose reads are over.  One: kt + 1 has landed, kt + 2 and kt + 3 may be in flight.  (Left alone, the compiler puts most reads behind the products and waits for each
        // few, and copies issued together keep a SIMD's two waves from the matrix pipe at the same time.)
        static_assert(GROUPS % NT == 0 && CPW <= NT, "a quarter's share");
        auto step = [&](const bf16x8 (&wv)[NT], const bf16x8 (&xv)[GROUPS], bf16x8 (&wn_)[NT], bf16x8 (&xn)[GROUPS], uint32_t k) {
            constexpr int Q = NT, PER = GROUPS / Q;        // quarters of a step
            const size_t from = (size_t)min(k + RING - 1, klast) * 1024;
            const uint32_t to = lds0 + ((k + RING - 1) % RING * KS + kh) * STAGE + wave * CPW * 1024;
            const unsigned char* st = mix_smem + ((k + 1) % RING * KS + kh) * STAGE;
#pragma unroll
            for (int q = 0; q < Q; q++) {
                __builtin_amdgcn_sched_barrier(0);
                if (q < CPW) lds_direct_load(to + q * 1024, src[q] + from, lane_off);
                __builtin_amdgcn_sched_barrier(0);
                wn_[q] = *reinterpret_cast<const bf16x8*>(st + w_off + q * 1024);
#pragma unroll
                for (int i = 0; i < PER; i++) xn[q * PER + i] = *reinterpret_cast<const bf16x8*>(st + x_off + (q * PER + i) * 1024);
#pragma unroll
                for (int i = 0; i < PER; i++)
#pragma unroll
                    for (int t = 0; t < NT; t++) acc[t][q * PER + i] = mix_mfma(wv[t], xv[q * PER + i], acc[t][q * PER + i]);
#pragma unroll
                for (int i = 0; i < 1 + PER; i++) {
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x008, NT * PER / (1 + PER), 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        constexpr bool PAIR = WN == 4;
        uint32_t kt = 0;
        for (; kt + 2 <= ktiles; kt += 2) {
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(CPW * (PAIR ? RING - 4 : RING - 3)) : "memory");
            step(w0, x0, w1, x1, kt);
            if constexpr (!PAIR) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(CPW * (RING - 3)) : "memory");
            step(w1, x1, w0, x0, kt + 1);
        }
        if (kt < ktiles) multiply(w0, x0);
    } else if constexpr (KS == 2) {
        bf16x8 w0[NT], x0[GROUPS], w1[NT], x1[GROUPS];
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(CPW * (RING - 2)) : "memory");
        read_ops(w0, x0, 0);
        // Step kt: everybody's copies of stage kt + 1 have landed, the copies of stage kt + 3 go to the slot of stage
        // kt - 1, whose last reads were waited for before step kt - 1 was multiplied; then the reads of stage kt + 1,
        // then the products of stage kt.  Two steps a turn, so that no register set is copied; a step past the end
        // reads a stage that holds a repeat of the last one and is not used.
        uint32_t kt = 0;
        for (; kt + 2 <= ktiles; kt += 2) {
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(CPW * (RING - 3)) : "memory");
            issue(kt + 3);
            read_ops(w1, x1, kt + 1);
            multiply(w0, x0);
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(CPW * (RING - 3)) : "memory");
            issue(kt + 4);
            read_ops(w0, x0, kt + 2);
            multiply(w1, x1);
        }
        if (kt < ktiles) multiply(w0, x0);
    } else
    for (uint32_t kt = 0; kt < ktiles; kt++) {
        // this wave's copies of stage kt have landed (those of kt + 1 may be in flight),
        // and everybody has finished reading stage kt - 1
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(CPW) : "memory");
        issue(kt + 2);
        bf16x8 wv[NT], xv[GROUPS];
        read_ops(wv, xv, kt);
        multiply(wv, xv);
        __builtin_amdgcn_sched_group_barrier(0x100, NT + GROUPS, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, NT * GROUPS, 0);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // the last steps' copies still target the ring

    if constexpr (KS == 2) {
        // (the rings are done with: every wave's copies have landed and, past the barrier, every wave's reads are over)
        static_assert((size_t)4 * NT * GROUPS * 1024 <= (size_t)RING * KS * STAGE, "the partial tiles fit the rings");
        f32x4* red = reinterpret_cast<f32x4*>(mix_smem) + (size_t)wave * NT * GROUPS * 64 + lane;
        lds_barrier();
        if (kh == 1) {
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int i = 0; i < GROUPS; i++) red[(t * GROUPS + i) * 64] = acc[t][i];
        }
        lds_barrier();
        if (kh == 1) return;
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int i = 0; i < GROUPS; i++) {
                const f32x4 o = red[(t * GROUPS + i) * 64];
#pragma unroll
                for (int j = 0; j < 4; j++) acc[t][i][j] += o[j];
            }
    }

    const uint32_t nt0 = nt_wg + wn * NT, group0 = g_wg + wr * GROUPS;
    if (nt0 >= a.ntiles || group0 >= a.groups) return;
    if (a.out >= kMixOutGated) {
#pragma unroll
        for (int t = 0; t < NT; t += 2)
#pragma unroll
            for (int i = 0; i < GROUPS; i++)
                mix_store_tile<false>(a, acc[t][i], acc[t + 1][i], nt0 + t, group0 + i, z, lane);
        return;
    }
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int i = 0; i < GROUPS; i++)
            mix_store_tile<false>(a, acc[t][i], acc[t][i], nt0 + t, group0 + i, z, lane);
}

}  // namespace wr
