// The layers of a decode step of one session in ONE launch.
//
// As separate launches a step of a 28-layer model is a chain of 140 (five a layer:
// Q/K/V product; row step + attention; output product; gate/up product; down
// product), each of which waits for the one before, fetches its arguments and its code,
// and only then asks for its weights: 4.5 .. 6.9 us each for 1 .. 2 us of HBM traffic.  Here one
// workgroup per CU stays for the whole step and the rows travel between workgroups
// as TAGGED values: eight bytes, the 32-bit value and the number of the step's layer it
// belongs to, stored through to memory.  A reader polls the values themselves until every
// tag is the one it waits for, so an exchange is one store and one load, no flag and no
// barrier between them (measured with nothing but the exchange, 256 workgroups: 1.4 us for
// 1024 values, 2.2 for 4096; with a flag per writer and the values read after it 3.6 and 4.2; a
// launch that reads its predecessor's row and writes another 3.1).
//
// A workgroup is eight waves.  Waves 0 .. 3 COMPUTE: they ask for the weights (or cache
// tiles) of the workgroup's next piece of work as soon as they are done with the
// last one, and hold them in registers until the row arrives.  Waves 4 .. 7 STAGE: they
// poll for the row, normalise it and write its operand terms to LDS.  The two kinds wait
// on counters of their own; a compute unit's loads still come back in the order they were
// made, so weights are asked for well ahead of the row or not until it is there.
//
//   piece      workgroups                        row in -> row out
//   qkv        a 16-output tile each             x [hidden], norm -> qkv
//   attention  KV head x key split               qkv -> partial rows (final ones if there is one split)
//   merge      a KV head each (staging waves)    partial rows -> attention rows
//   o          a tile each                       attention rows (+ x) -> x2 [hidden]
//   gate/up    a pair of tiles each              x2, norm -> act [ffn]
//   down       a tile each                       act (+ x2) -> x
//
// What bounds it: the chain of exchanges.  28 layers, hidden 1024, 16/8 heads, ffn 3072, at 60 keys: 464 us in the
// launch, 16.6 a layer (140 launches: 770), for 4.7 us of weights from HBM: five exchanges of 0.8 to 1.4 us (store, load,
// and half a load's trip until the next look; a sixth where keys are split), four times 0.8 from row to terms and 0.6 from
// terms to the next row, and 3.5 us in the attention.  (488 and 17.4 before a layer's norm weights were asked for behind
// attention and its first keys ahead of the Q/K/V weights: the Q/K/V row's exchange took 1.8 to 3.0 us.)
//
// A row's buffer is written once a layer.  Whoever writes it again has, through the rows in
// between, waited for every reader of the last layer's values: each piece reads its row before it
// writes, and a row is complete only when all of its pieces have written.
//
// Values, scales and the order of every sum are those of proj_row1_kernel and
// decode_mfma_kernel<128, true>, so the bits are those of the chain of launches.
//
// All workgroups have to run at once: one per CU at most, the host makes sure that no
// second such launch of this process is on the device, and every wait ends at a
// deadline by the clock (another process may hold the CUs).  After it nothing waits any more,
// the launch runs to its end on whatever is there, the host is told, and takes the chain.
#pragma once

#include "kernels_decode.hip.h"
#include "kernels_proj.hip.h"

namespace wr {

constexpr int kStepThreads = 512;
constexpr uint32_t kStepTiles = 24;          // weight tiles a wave holds: inputs up to 3072 (gated: 1536)
constexpr uint32_t kStepLimitTicks = 5000000;    // 50 ms of the 100 MHz clock; a step takes about half a millisecond

// (the device's own memory: an address read from memory is otherwise taken to be any, and a flat load is
// counted with LDS traffic, whose barriers would then wait for weights)
typedef const __attribute__((address_space(1))) half8* StepWeights;
typedef const __attribute__((address_space(1))) f32x4* StepNorm;

struct StepLayer {
    const half8* wqkv;
    const half8* wo;
    const half8* wgu;
    const half8* wdown;
    const float* attn_norm;
    const float* ffn_norm;
    const float* q_norm;     // or null, with k_norm
    const float* k_norm;
};

struct StepArgs {
    const StepLayer* layers;
    const float* x0;         // [hidden], plain: written before this launch
    float* y;                // [hidden], plain: the last layer's row
    const float* cos_sin;    // [n_rot][2], or null
    uint8_t* slab;           // cache: K of layer l at 2 l side, Vt at (2 l + 1) side
    u32x4* x;                // tagged rows (step_unit gives the places), all but qkv in kStepCopies
    u32x4* qkv;
    u32x4* attn;
    u32x4* x2;
    u32x4* act;
    uint64_t* part;          // [nq][n_splits][128] tagged
    uint64_t* part_ml;       // [nq][n_splits][2] tagged
    uint32_t* expired;       // host memory: set when a wait met its deadline
    DecodeSession s;         // (k, vt: unused)
    uint64_t side;
    uint32_t n_layers, hidden, ffn, nq, nkv, n_rot;
    uint32_t tag0;           // tag of layer l: tag0 + l
    uint32_t limit;          // ticks until every wait ends
    float eps, qscale;
};

// Tagged values: the 16 values of a product's tile are one 128-byte line, written whole in two stores of
// 64 bytes (a line that eight-byte stores or several tiles share takes a microsecond longer to be seen).  Values
// 4 j .. 4 j + 3 (quad j of the tile) are the 16-byte units j and 4 + j of the line, two values and
// their tags each.
__host__ __device__ __forceinline__ uint32_t step_unit(uint32_t quad, uint32_t p) { return (quad >> 2) * 8 + p * 4 + (quad & 3); }
__host__ __device__ __forceinline__ uint32_t step_row_units(uint32_t n) { return n / 2; }

// A row that every workgroup polls is kept in copies, which the workgroups share out: the requests of 256 of them
// for the same 64 lines queue in the few memory channels that those lie in (a trip took 1.2 us).
constexpr uint32_t kStepCopies = 8;

__device__ __forceinline__ uint32_t step_copy(uint32_t n) { return blockIdx.x % kStepCopies * step_row_units(n); }

__device__ __forceinline__ uint64_t step_tagged(float v, uint32_t tag) { return (uint64_t)tag << 32 | __float_as_uint(v); }
__device__ __forceinline__ void step_put(uint64_t* p, float v, uint32_t tag)
{
    __hip_atomic_store(p, step_tagged(v, tag), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t step_get(const uint64_t* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Two tagged values as one 16-byte load past what the XCD's own L2 holds (sc1); each aligned
// eight bytes of it arrive whole, and carry a tag of their own.
__device__ __forceinline__ u32x4 step_get_unit(__amdgpu_buffer_rsrc_t row, uint32_t unit)
{
    return __builtin_amdgcn_raw_buffer_load_b128(row, (int)(unit * 16), 0, 16);
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t step_row(const u32x4* p, uint32_t n)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<u32x4*>(p), 0, (int)(step_row_units(n) * 16), 0x00020000);
}

// A wait's own end: true when the deadline has passed (and the host is told).  Looked at every sixteenth time.
__device__ __forceinline__ bool step_late(const StepArgs& a, uint64_t deadline, uint32_t& tries)
{
    if ((++tries & 15) != 0 || __builtin_amdgcn_s_memrealtime() < deadline) return false;
    __hip_atomic_store(a.expired, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    return true;
}

// Staging lane: the quads q[i] of a tagged row.  (Two requests under way at a time, half a trip apart, were no faster:
// the one that is not needed any more holds up whatever comes next.)
template <int N>
__device__ __forceinline__ void step_poll(const StepArgs& a, float (&v)[N][4], __amdgpu_buffer_rsrc_t row, const uint32_t (&q)[N],
                                          uint32_t tag, uint64_t deadline)
{
    u32x4 u[N][2];
    for (uint32_t tries = 0;;) {
        bool ok = true;
        asm volatile("" ::: "memory");                       // (asked for again every time)
#pragma unroll
        for (int i = 0; i < N; i++)
#pragma unroll
            for (int p = 0; p < 2; p++) u[i][p] = step_get_unit(row, step_unit(q[i], p));
#pragma unroll
        for (int i = 0; i < N; i++)
#pragma unroll
            for (int p = 0; p < 2; p++) ok = ok && u[i][p][1] == tag && u[i][p][3] == tag;
        if (__all(ok) || step_late(a, deadline, tries)) break;
    }
#pragma unroll
    for (int i = 0; i < N; i++)
#pragma unroll
        for (int p = 0; p < 2; p++) {
            v[i][2 * p] = __uint_as_float(u[i][p][0]);
            v[i][2 * p + 1] = __uint_as_float(u[i][p][2]);
        }
}

constexpr int kStepHeads = (kMaxGroupMfma + 2 + 3) / 4;     // heads of an attention piece (Q's, K, V) to a staging wave

struct StepShared {
    f32x4 part[6 * 64];                                     // sums of compute waves 1 .. 3
    float sum[8];
    float max[4];
    float scale;
    alignas(16) float resid[16];
    _Float16 q[16][128 + 8];
    DecodeNewRow<128> row;
    float o[kDecodeWaves][2 * kMaxGroupMfma][128 + 4];       // a head's hi column, G on its lo column
    float m[kDecodeWaves][kMaxGroupMfma];
    float l[kDecodeWaves][kMaxGroupMfma];
    alignas(16) float head[4][kStepHeads][128];              // a staging wave's heads of the Q/K/V row
};

// What a staging lane holds of a row: quad i, of a chunk that others may not have.
__device__ __forceinline__ uint32_t step_chunk(uint32_t t, int i)
{
    const uint32_t lane = t & 63, wave = t >> 6;
    return (2 * i + (wave >> 1)) * 64 + (lane >> 1) * 2 + (wave & 1);
}
__device__ __forceinline__ uint32_t step_quad(uint32_t t, int i, uint32_t nchunks) { return min(step_chunk(t, i), nchunks - 1) * 2 + (t & 1); }

// Norm weights are asked for behind the attention ahead of their rows: a wave's loads come back in the order they were made, and the first look at
// a row would wait for the trip to memory that weights nobody has read yet take (1.7 us).
__device__ __forceinline__ void step_norm_weights(f32x4 (&w)[2], const float* norm, uint32_t t, uint32_t hidden)
{
#pragma unroll
    for (int i = 0; i < 2; i++) w[i] = ((StepNorm)norm)[step_quad(t, i, hidden / 8)];
}

// Staging waves: a row's operand terms, as proj_row1_kernel forms them (t = 0 .. 255 over the four
// waves).  `plain`: the row as plain values instead of a tagged one.  resid: the row of which a product's tile adds
// 16 values (tagged, or plain), or null.
//
// A lane takes four values of a chunk of eight, its neighbour the other four: with eight to a
// lane half of the lanes had none of a row of 1024, and the arithmetic from the row to its terms took 1.0 us.
// The sum of squares keeps its order: down a chunk, then a tree over 64 chunks whose last
// step adds the odd ones' sum to the even ones', which is why waves w and w ^ 1 take the even and the odd chunks of the
// same 64, then the sums of 64 chunks in pairs.
template <int N>
__device__ __forceinline__ void step_stage(const StepArgs& a, StepShared& sh, half8* sfrag, uint32_t t, const u32x4* tagged,
                                           const float* plain, uint32_t K, bool norm, const f32x4 (&weights)[2], uint32_t tag,
                                           uint64_t deadline, const u32x4* resid, const float* resid_plain, uint32_t resid_tag, uint32_t tile)
{
    const uint32_t nchunks = K / 8;
    const uint32_t lane = t & 63, wave = t >> 6;
    uint32_t q[N];
    bool has[N];
#pragma unroll
    for (int i = 0; i < N; i++) {
        q[i] = step_quad(t, i, nchunks);
        has[i] = step_chunk(t, i) < nchunks;
    }
    float r = 0.f;                                           // the residual's values were there before this row could be made
    if (wave == 3 && (resid || resid_plain) && lane < 16) {
        const uint32_t k = tile * 16 + lane;
        if (resid_plain) {
            r = resid_plain[k];
        } else {
            const uint64_t* p = reinterpret_cast<const uint64_t*>(resid + step_copy(a.hidden) + step_unit(k >> 2, (k >> 1) & 1)) + (k & 1);
            uint64_t w;
            for (uint32_t tries = 0;;) {
                w = step_get(p);
                if (__all((uint32_t)(w >> 32) == resid_tag) || step_late(a, deadline, tries)) break;
            }
            r = __uint_as_float((uint32_t)w);
        }
    }
    float v[N][4];
    if (plain) {
#pragma unroll
        for (int i = 0; i < N; i++) {
            const f32x4 x = *reinterpret_cast<const f32x4*>(plain + q[i] * 4);
#pragma unroll
            for (int j = 0; j < 4; j++) v[i][j] = has[i] ? x[j] : 0.f;
        }
    } else {
        step_poll<N>(a, v, step_row(tagged + step_copy(K), K), q, tag, deadline);
#pragma unroll
        for (int i = 0; i < N; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) v[i][j] = has[i] ? v[i][j] : 0.f;
    }
    if (norm) {
#pragma unroll
        for (int i = 0; i < (N < 2 ? N : 2); i++) {          // (a row that is normalised has 2048 values at most)
            float ss = 0.f;
#pragma unroll
            for (int j = 0; j < 4; j++) ss = fmaf(v[i][j], v[i][j], ss);
            ss = wave_xor_f32(ss, 1);                        // the odd lanes go on where the even ones have ended
#pragma unroll
            for (int j = 0; j < 4; j++) ss = fmaf(v[i][j], v[i][j], ss);
#pragma unroll
            for (int off = 32; off >= 2; off >>= 1) ss += wave_xor_f32(ss, off);
            if (lane == 1) sh.sum[i * 4 + wave] = ss;
        }
        lds_barrier();
        float ss = (sh.sum[0] + sh.sum[1]) + (sh.sum[2] + sh.sum[3]);
        if (N > 1) ss += (sh.sum[4] + sh.sum[5]) + (sh.sum[6] + sh.sum[7]);
        const float inv_rms = 1.0f / sqrtf(ss / (float)K + a.eps);
#pragma unroll
        for (int i = 0; i < (N < 2 ? N : 2); i++)
#pragma unroll
            for (int j = 0; j < 4; j++) v[i][j] = v[i][j] * inv_rms * weights[i][j];
    }
    float mx = 0.f;
#pragma unroll
    for (int i = 0; i < N; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) mx = fmaxf(mx, fabsf(v[i][j]));
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, wave_xor_f32(mx, off));
    if (lane == 0) sh.max[wave] = mx;
    lds_barrier();
    mx = fmaxf(fmaxf(sh.max[0], sh.max[1]), fmaxf(sh.max[2], sh.max[3]));
    uint32_t ex = (__float_as_uint(mx) >> 23) & 0xFFu;
    if (ex == 0 || ex == 0xFF) ex = 127;
    if (ex > 253) ex = 253;
    if (t == 0) sh.scale = __uint_as_float(ex << 23);
    if (wave == 3 && lane < 16) sh.resid[lane] = r;
    const float inv = __uint_as_float((254u - ex) << 23);
    half4* terms = reinterpret_cast<half4*>(sfrag);          // of a chunk: hi of its eight inputs, then lo
#pragma unroll
    for (int i = 0; i < N; i++) {
        half4 hi, lo;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float sv = v[i][j] * inv;
            _Float16 h = (_Float16)sv;
            if (fabsf((float)h) < 6.103515625e-05f) h = (_Float16)0.0f;      // 2^-14
            hi[j] = h;
            lo[j] = (_Float16)((sv - (float)h) * kProjLoScale);
        }
        if (has[i]) {
            terms[(q[i] >> 1) * 4 + (q[i] & 1)] = hi;
            terms[(q[i] >> 1) * 4 + 2 + (q[i] & 1)] = lo;
        }
    }
    lds_barrier();                                           // the terms are there
    lds_barrier();                                           // the compute waves have read them
}

// Compute waves: a product's tile (NT = 2: a gate's and its values') against the staged row, NB batches of four
// k-steps to a wave.  norm: the staging waves' barrier more before the terms are there.  Wave 0: the sums in acc, the
// row's scale and, lane 16 g, the residual's values 4 g .. + 3.
template <int NT, int NB>
__device__ __forceinline__ void step_product_of(StepShared& sh, const half8* sfrag, f32x4 (&acc)[NT], float& scale, f32x4& resid,
                                                StepWeights w, uint32_t tile0, uint32_t tile1, bool norm, int lane, uint32_t wave)
{
    constexpr uint32_t KS = NB * 4, ktiles = KS * 4;
    const uint32_t k0 = wave * KS;
    StepWeights wp[2] = {w + ((size_t)tile0 * ktiles + k0) * 64, w + ((size_t)tile1 * ktiles + k0) * 64};
    half8 wv[KS][NT];
#pragma unroll
    for (uint32_t u = 0; u < KS; u++)
#pragma unroll
        for (int tt = 0; tt < NT; tt++) wv[u][tt] = __builtin_nontemporal_load(wp[tt] + u * 64 + lane);
    // columns without a row are zeros (made ahead of the wait: 64 lanes reading them took down's 24 steps 0.3 us)
    u32x4 xb[2][4];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        xb[i / 4][i % 4] = u32x4{0, 0, 0, 0};
        asm volatile("" : "+v"(xb[i / 4][i % 4]));
    }
    const int c = lane & 15, g = lane >> 4;
    const bool has = (c & 7) == 0;
    const u32x4* my = reinterpret_cast<const u32x4*>(sfrag) + (size_t)k0 * 8 + g * 2 + (c >> 3);
    if (norm) lds_barrier();
    lds_barrier();
    lds_barrier();
    const auto terms = [&](uint32_t batch) {
        if (has) {
#pragma unroll
            for (uint32_t u = 0; u < 4; u++) xb[batch & 1][u] = my[(batch * 4 + u) * 8];
        }
    };
    terms(0);
    scale = sh.scale;
    resid = *reinterpret_cast<const f32x4*>(&sh.resid[4 * g]);
#pragma unroll
    for (int tt = 0; tt < NT; tt++) acc[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (uint32_t n = 0; n < NB; n++) {
        if (n + 1 < NB) terms(n + 1);
#pragma unroll
        for (uint32_t u = 0; u < 4; u++)
#pragma unroll
            for (int tt = 0; tt < NT; tt++)
                acc[tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv[n * 4 + u][tt], __builtin_bit_cast(half8, xb[n & 1][u]), acc[tt], 0, 0, 0);
    }
    if (wave > 0 && has) {                                   // (the other columns are of no row)
#pragma unroll
        for (int tt = 0; tt < NT; tt++) sh.part[((wave - 1) * NT + tt) * 64 + lane] = acc[tt];
    }
    lds_barrier();
    if (wave == 0) {
        f32x4 o[3][NT];
#pragma unroll
        for (int p = 0; p < 3; p++)
#pragma unroll
            for (int tt = 0; tt < NT; tt++) o[p][tt] = sh.part[(p * NT + tt) * 64 + lane];
#pragma unroll
        for (int p = 0; p < 3; p++)
#pragma unroll
            for (int tt = 0; tt < NT; tt++)
#pragma unroll
                for (int i = 0; i < 4; i++) acc[tt][i] += o[p][tt][i];
#pragma unroll
        for (int tt = 0; tt < NT; tt++) acc[tt] = proj_join_terms(acc[tt]);
    } else {
        __builtin_amdgcn_s_sleep(10);                        // wave 0's results go out before the next weights are asked for
    }
}

template <int NT>
__device__ __forceinline__ void step_product(StepShared& sh, const half8* sfrag, f32x4 (&acc)[NT], float& scale, f32x4& resid,
                                             StepWeights w, uint32_t tile0, uint32_t tile1, uint32_t n_in, bool norm, int lane,
                                             uint32_t wave)
{
    const auto run = [&](auto batches) {
        step_product_of<NT, decltype(batches)::value>(sh, sfrag, acc, scale, resid, w, tile0, tile1, norm, lane, wave);
    };
    switch (n_in / 512) {
    case 1: return run(std::integral_constant<int, 1>());
    case 2: return run(std::integral_constant<int, 2>());
    case 3: return run(std::integral_constant<int, 3>());
    }
    if constexpr (NT == 1) switch (n_in / 512) {
        case 4: return run(std::integral_constant<int, 4>());
        case 5: return run(std::integral_constant<int, 5>());
        case 6: return run(std::integral_constant<int, 6>());
        }
}

// Wave 0: the 16 outputs of a tile (lane 16 g holds 4 g .. + 3) into the row's copies, all in one store: lane 8 c + u
// writes unit u of copy c.  (Through to memory: sc1.)
__device__ __forceinline__ void step_publish(u32x4* row, uint32_t n, uint32_t copies, uint32_t tile, int lane, const f32x4& r, uint32_t tag)
{
    const int from = (lane & 3) * 64;                        // lane 16 j of quad j, as a byte address
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = __int_as_float(__builtin_amdgcn_ds_bpermute(from, __float_as_int(r[i])));
    const bool p = (lane & 4) != 0;
    const u32x4 unit = u32x4{__float_as_uint(p ? v[2] : v[0]), tag, __float_as_uint(p ? v[3] : v[1]), tag};
    const uint32_t copy = (uint32_t)lane >> 3;
    const __amdgpu_buffer_rsrc_t at = __builtin_amdgcn_make_buffer_rsrc(row, 0, (int)(copies * step_row_units(n) * 16), 0x00020000);
    if (copy < copies)
        __builtin_amdgcn_raw_buffer_store_b128(unit, at, (int)((copy * step_row_units(n) + tile * 8 + (lane & 7)) * 16), 0, 16);
}

// A value of the attention rows, into all copies.
__device__ __forceinline__ void step_put_copies(const StepArgs& a, uint32_t at, float v, uint32_t tag)
{
    uint64_t* p = reinterpret_cast<uint64_t*>(a.attn) + at;
#pragma unroll
    for (uint32_t c = 0; c < kStepCopies; c++) step_put(p + (size_t)c * a.nq * 128, v, tag);
}

// The element of a head's 128 values that is the i-th of its tagged values.
__device__ __forceinline__ uint32_t step_head_dim(uint32_t i) { return (i & ~15u) + ((i >> 1) & 3) * 4 + ((i >> 3) & 1) * 2 + (i & 1); }

// Attention of one (KV head, key split), compute waves; as decode_mfma_kernel<128, true>.
// `fa`: the wave's first tile, asked for (step_first_tile) ahead of the layer.
__device__ __forceinline__ void step_first_tile(const StepArgs& a, DecodeFrag<128>& fa, uint32_t kvh, uint32_t split, const uint16_t* kc,
                                                const uint16_t* vc, int lane, uint32_t wave)
{
    const TileRange tr = split_tiles(a.s, split);
    load_frag<128>(fa, kc + (size_t)kvh * a.s.ctx_pad * 128, vc + (size_t)kvh * (a.s.ctx_pad / kVBlock) * 128 * kVBlock,
                   min(tr.t_begin + wave, tr.t_end - 1), lane);
}

__device__ __forceinline__ void step_attend(const StepArgs& a, StepShared& sh, DecodeFrag<128>& fa, uint32_t kvh, uint32_t split,
                                            const uint16_t* kc, const uint16_t* vc, uint32_t tag, int lane, uint32_t wave)
{
    constexpr int HD = 128;
    const DecodeSession& S = a.s;
    const int n = lane & 15, g = lane >> 4;
    const int G = (int)(a.nq / a.nkv);
    const TileRange tr = split_tiles(S, split);
    const uint16_t* kbase = kc + (size_t)kvh * S.ctx_pad * HD;
    const uint16_t* vtbase = vc + (size_t)kvh * (S.ctx_pad / kVBlock) * HD * kVBlock;
    const uint32_t new_tile = (S.seq_k - 1) / kTileKeys;
    const bool owner = new_tile >= tr.t_begin && new_tile < tr.t_end;
    const uint32_t patch_tile = (owner && (new_tile - tr.t_begin) % kDecodeWaves == wave) ? new_tile : 0xFFFFFFFFu;
    uint32_t t = tr.t_begin + wave;
    lds_barrier();                                           // Q^T and the new row are in LDS

    const int col_kind = (n < G) ? 0 : ((n < 2 * G) ? 1 : 2);
    const int partner = (n < G) ? lane + G : ((n < 2 * G) ? lane - G : lane);
    const int partner_addr = partner * 4;
    DecodeState<HD> st;
#pragma unroll
    for (int dt = 0; dt < HD / 16; dt++) st.o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    st.m = -INFINITY;
    st.l = 0.f;
    const _Float16* qrow = &sh.q[n][g * 8];
    if (t < tr.t_end) {
        f32x4 c[2];
        while (t + kDecodeWaves < tr.t_end) {
            asm volatile("" ::: "memory");                   // keeps the Q^T reads inside the loop
            tile_scores_lds<HD>(c, fa, qrow);
            load_frag_k<HD>(fa, kbase, t + kDecodeWaves, lane);
            tile_update<HD>(st, fa, c, t, S.key_lo, S.seq_k, lane, partner_addr, col_kind);
            load_frag_v<HD>(fa, vtbase, t + kDecodeWaves, lane);
            t += kDecodeWaves;
        }
        if (t == patch_tile) patch_new_row<HD>(fa, sh.row, (S.seq_k - 1) % kTileKeys, lane);
        tile_scores_lds<HD>(c, fa, qrow);
        tile_update<HD>(st, fa, c, t, S.key_lo, S.seq_k, lane, partner_addr, col_kind);
    }
    st.l += wave_xor_f32(st.l, 16);
    st.l += wave_xor_f32(st.l, 32);
    if (n < 2 * G) {                                         // (a head's two columns are added below)
#pragma unroll
        for (int dt = 0; dt < HD / 16; dt++) *reinterpret_cast<f32x4*>(&sh.o[wave][n][dt * 16 + 4 * g]) = st.o[dt];
        if (n < G && g == 0) {
            sh.m[wave][n] = st.m;
            sh.l[wave][n] = st.l;
        }
    }
    lds_barrier();
    for (uint32_t idx = wave * 64 + lane; idx < (uint32_t)G * HD; idx += kDecodeThreads) {
        const uint32_t h = idx / HD, i = idx % HD, d = step_head_dim(i);
        float M = sh.m[0][h];
#pragma unroll
        for (int w = 1; w < kDecodeWaves; w++) M = fmaxf(M, sh.m[w][h]);
        float acc = 0.f, L = 0.f;
#pragma unroll
        for (int w = 0; w < kDecodeWaves; w++) {
            const float fct = fast_exp2(sh.m[w][h] - M);
            acc += (sh.o[w][h][d] + sh.o[w][h + G][d]) * fct;
            L += sh.l[w][h] * fct;
        }
        const uint32_t head = kvh * G + h;
        if (S.n_splits == 1) {
            step_put_copies(a, head * HD + i, (L > 0.f) ? acc / L : 0.f, tag);
        } else {
            const size_t pi = (size_t)head * S.n_splits + split;
            step_put(a.part + pi * HD + i, acc, tag);
            if (i == 0) {
                step_put(a.part_ml + pi * 2, M, tag);
                step_put(a.part_ml + pi * 2 + 1, L, tag);
            }
        }
    }
}

// The head of an attention piece that a staging lane has its part of: Q's 0 .. G - 1, then K, then V, dealt to the waves
// in turn, eight lanes each.
constexpr uint32_t kStepNoHead = 0xFFFFFFFFu;
__device__ __forceinline__ uint32_t step_head_slot(uint32_t t, uint32_t G)
{
    const uint32_t octet = (t & 63) >> 3, slot = octet * 4 + (t >> 6);
    return octet < (uint32_t)kStepHeads && slot < G + 2 ? slot : kStepNoHead;
}

// The norm's weights (a layer ahead, as above) and the rotation of a staging lane's part of its head.  Asked for whether
// they are used or not, from an address that is valid.
__device__ __forceinline__ void step_head_weights(const StepArgs& a, Row8Loads<2>& rl, const StepLayer& ly, uint32_t t)
{
    const uint32_t G = a.nq / a.nkv;
    const float* nw = step_head_slot(t, G) == G ? ly.k_norm : ly.q_norm;
    const StepNorm w = (StepNorm)(nw ? nw : a.x0);
#pragma unroll
    for (int c = 0; c < 2; c++) {
        rl.w[c][0] = w[c * 16 + (t & 7) * 2];
        rl.w[c][1] = w[c * 16 + (t & 7) * 2 + 1];
    }
}
__device__ __forceinline__ void step_head_turn(const StepArgs& a, Row8Loads<2>& rl, uint32_t t)
{
    const StepNorm cs = (StepNorm)(a.cos_sin ? a.cos_sin : a.x0);
    const uint32_t j0 = a.cos_sin ? min((t & 7) * 8, a.n_rot - 8) : 0u;
#pragma unroll
    for (int q = 0; q < 4; q++) rl.t[0][q] = cs[j0 / 2 + q];
}

// The row step of an attention piece, staging waves (t = 0 .. 255): Q heads into the Q^T operand, and in the workgroup
// whose keys hold the new position K and V into the cache and into LDS.
__device__ __forceinline__ void step_attend_stage(const StepArgs& a, StepShared& sh, Row8Loads<2>& rl, bool norm, uint32_t kvh, uint32_t split,
                                                  uint16_t* kc, uint16_t* vc, uint32_t tag, uint32_t t, uint64_t deadline)
{
    constexpr int HD = 128, NJ = HD / 64;
    const DecodeSession& S = a.s;
    const int G = (int)(a.nq / a.nkv);
    const TileRange tr = split_tiles(S, split);
    const uint32_t new_pos = S.seq_k - 1, new_tile = new_pos / kTileKeys;
    const bool owner = new_tile >= tr.t_begin && new_tile < tr.t_end;
    const uint32_t lane = t & 63, wave = t >> 6, part = t & 7, slot = step_head_slot(t, G);
    const bool slot_q = slot < (uint32_t)G, slot_k = owner && slot == (uint32_t)G, slot_v = owner && slot == (uint32_t)G + 1;
    // A wave asks for each of its heads with one load, 1024 bytes side by side, and takes them apart through LDS.
    const __amdgpu_buffer_rsrc_t row = step_row(a.qkv, (a.nq + 2 * a.nkv) * HD);
    u32x4 u[kStepHeads];
    const auto used = [&](int i) { return i * 4 + wave < (uint32_t)(owner ? G + 2 : G); };      // (the same in all lanes)
    for (uint32_t tries = 0;;) {
        bool ok = true;
        asm volatile("" ::: "memory");                       // (asked for again every time)
#pragma unroll
        for (int i = 0; i < kStepHeads; i++) {
            const uint32_t sl = i * 4 + wave;
            const uint32_t head = sl < (uint32_t)G ? kvh * G + sl : sl == (uint32_t)G ? a.nq + kvh : a.nq + a.nkv + kvh;
            u[i] = u32x4{0, tag, 0, tag};
            if (used(i)) u[i] = step_get_unit(row, head * 64 + lane);
        }
#pragma unroll
        for (int i = 0; i < kStepHeads; i++) ok = ok && u[i][1] == tag && u[i][3] == tag;
        if (__all(ok) || step_late(a, deadline, tries)) break;
    }
#pragma unroll
    for (int i = 0; i < kStepHeads; i++) {
        float2 two{__uint_as_float(u[i][0]), __uint_as_float(u[i][2])};
        *reinterpret_cast<float2*>(&sh.head[wave][i][(lane >> 3) * 16 + (lane & 3) * 4 + (lane >> 2 & 1) * 2]) = two;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // (its own wave's)
    const float* mine = sh.head[wave][min(lane >> 3, (uint32_t)kStepHeads - 1)] + part * 8;
#pragma unroll
    for (int c = 0; c < NJ; c++)
#pragma unroll
        for (int e = 0; e < 2; e++) rl.x[c][e] = *reinterpret_cast<const f32x4*>(mine + c * 64 + e * 4);
    float x[NJ][8];
    row8_head_finish<NJ>(x, rl, norm && !slot_v, false, a.eps, part, a.cos_sin != nullptr && !slot_v, a.n_rot);
    if (slot_q) {
#pragma unroll
        for (int c = 0; c < NJ; c++)
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int d = c * 64 + (int)part * 8 + e;
                _Float16 hi, lo;
                q_hi_lo(x[c][e], a.qscale, hi, lo);
                sh.q[slot][d] = hi;
                sh.q[slot + G][d] = lo;
            }
    }
    u32x4 packed[NJ];                                        // K or V as the cache holds them
    if (slot_k || slot_v) {
#pragma unroll
        for (int c = 0; c < NJ; c++) {
#pragma unroll
            for (int e = 0; e < 4; e++)
                packed[c][e] = (uint32_t)f32_to_f16_trunc(x[c][2 * e]) | ((uint32_t)f32_to_f16_trunc(x[c][2 * e + 1]) << 16);
            *reinterpret_cast<u32x4*>(&(slot_k ? sh.row.k : sh.row.v)[c * 64 + part * 8]) = packed[c];
        }
    }
    lds_barrier();                                           // Q^T and the new row are in LDS
    lds_barrier();                                           // the waves' partial rows are
    if (slot_k) {
#pragma unroll
        for (int c = 0; c < NJ; c++) *reinterpret_cast<u32x4*>(kc + k_offset(kvh, S.ctx_pad, new_pos, c * 64 + part * 8, HD)) = packed[c];
    } else if (slot_v) {
#pragma unroll
        for (int c = 0; c < NJ; c++)
#pragma unroll
            for (int e = 0; e < 8; e++)
                vc[vt_offset(kvh, S.ctx_pad, new_pos, c * 64 + part * 8 + e, HD)] = (uint16_t)(packed[c][e >> 1] >> (16 * (e & 1)));
    }
}

// Staging waves: the rows of a KV head's group from their partial rows; as merge_in_regs.
__device__ __forceinline__ void step_merge(const StepArgs& a, uint32_t kvh, uint32_t tag, uint32_t t, uint64_t deadline)
{
    constexpr uint32_t HD = 128, N = kMergeInRegs;
    const uint32_t G = a.nq / a.nkv, n_splits = a.s.n_splits;
    for (uint32_t idx = t; idx < G * HD; idx += 256) {
        const uint32_t h = idx / HD, i = idx % HD;
        const uint64_t* pv = a.part + (size_t)(kvh * G + h) * n_splits * HD + i;
        const uint64_t* pm = a.part_ml + (size_t)(kvh * G + h) * n_splits * 2;
        float v[N], m[N], l[N];
        for (uint32_t tries = 0;;) {
            bool ok = true;
            uint64_t wv[N], wm[N], wl[N];
#pragma unroll
            for (uint32_t k = 0; k < N; k++) {
                wv[k] = wm[k] = wl[k] = (uint64_t)tag << 32;
                if (k < n_splits) {
                    wv[k] = step_get(pv + k * HD);
                    wm[k] = step_get(pm + k * 2);
                    wl[k] = step_get(pm + k * 2 + 1);
                }
            }
#pragma unroll
            for (uint32_t k = 0; k < N; k++) {
                ok = ok && (uint32_t)(wv[k] >> 32) == tag && (uint32_t)(wm[k] >> 32) == tag && (uint32_t)(wl[k] >> 32) == tag;
                v[k] = __uint_as_float((uint32_t)wv[k]);
                m[k] = __uint_as_float((uint32_t)wm[k]);
                l[k] = __uint_as_float((uint32_t)wl[k]);
            }
            if (__all(ok) || step_late(a, deadline, tries)) break;
        }
        step_put_copies(a, (kvh * G + h) * HD + i, merge_partials<N>(v, m, l, n_splits), tag);
    }
}

constexpr uint32_t kStepQkv = 0, kStepAttend = 1, kStepOut = 2, kStepGateUp = 3, kStepDown = 4;

// A layer's addresses, through the scalar cache (nothing writes them while a model lives).
__device__ __forceinline__ StepLayer step_layer(const StepArgs& a, uint32_t L)
{
    typedef const __attribute__((address_space(4))) uint64_t* Words;
    const Words w = (Words)(uintptr_t)(a.layers + L);
    StepLayer y;
    y.wqkv = (const half8*)w[0];
    y.wo = (const half8*)w[1];
    y.wgu = (const half8*)w[2];
    y.wdown = (const half8*)w[3];
    y.attn_norm = (const float*)w[4];
    y.ffn_norm = (const float*)w[5];
    y.q_norm = (const float*)w[6];
    y.k_norm = (const float*)w[7];
    return y;
}

__global__ __launch_bounds__(kStepThreads, 2) void step_layers_kernel(const StepArgs a)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char step_smem[];
    half8* sfrag = reinterpret_cast<half8*>(step_smem);      // [inputs / 8][2]: hi, lo of a chunk
    __shared__ StepShared sh;
    const int lane = threadIdx.x & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint64_t deadline = __builtin_amdgcn_s_memrealtime() + a.limit;
    // The workgroup's pieces, at most one of a kind (the host has seen to it).  Pairs of the gate/up product
    // begin behind the tiles of the output and down products, which share workgroups: those have that long to
    // ask for their weights, the longest.  Attention takes workgroups from the end.
    const uint32_t b = blockIdx.x, grid = gridDim.x;
    const uint32_t qd = a.nq * 128, width = (a.nq + 2 * a.nkv) * 128;
    const uint32_t htiles = a.hidden / 16;
    const uint32_t behind = b >= htiles ? b - htiles : b + grid - htiles;
    const uint32_t item = grid - 1 - b;
    const bool has_qkv = b < width / 16, has_o = b < htiles, has_gu = behind < a.ffn / 16;
    const bool has_attn = item < a.nkv * a.s.n_splits, has_merge = a.s.n_splits > 1 && behind < a.nkv;
    const uint32_t pieces = (has_qkv ? 1u << kStepQkv : 0u) | (has_attn || has_merge ? 1u << kStepAttend : 0u) |
                            (has_o ? 1u << kStepOut | 1u << kStepDown : 0u) | (has_gu ? 1u << kStepGateUp : 0u);
    const uint32_t kvh = item % a.nkv, split = item / a.nkv;

    for (uint32_t i = threadIdx.x; i < 16 * 136 / 8; i += kStepThreads) reinterpret_cast<half8*>(&sh.q[0][0])[i] = half8{};
    if (threadIdx.x < 8) sh.sum[threadIdx.x] = 0.f;
    lds_barrier();
    if (wave >= 4) {
        StepLayer next = step_layer(a, 0);
        f32x4 attn_w[2], ffn_w[2] = {};
        Row8Loads<2> rl;
        step_norm_weights(attn_w, next.attn_norm, threadIdx.x - 256, a.hidden);
        step_head_turn(a, rl, threadIdx.x - 256);
        step_head_weights(a, rl, next, threadIdx.x - 256);
        for (uint32_t L = 0; L < a.n_layers; L++) {
            const StepLayer ly = next;
            next = step_layer(a, min(L + 1, a.n_layers - 1));
            const uint32_t tag = a.tag0 + L;
            const float* x0 = L == 0 ? a.x0 : nullptr;       // the row ahead of the first layer; later ones bear the tag before
            uint16_t* kc = reinterpret_cast<uint16_t*>(a.slab + 2 * L * a.side);
            uint16_t* vc = reinterpret_cast<uint16_t*>(a.slab + (2 * L + 1) * a.side);
            for (uint32_t piece = kStepQkv; piece <= kStepDown; piece++) {
                uint32_t t = threadIdx.x - 256;
                asm volatile("" : "+v"(t));                  // what a piece derives from the lane is not kept through the others
                if (piece == kStepOut) {                     // (attention's row, or a layer's first, would come in behind them)
                    if (has_gu) step_norm_weights(ffn_w, ly.ffn_norm, t, a.hidden);
                    if (has_qkv) step_norm_weights(attn_w, next.attn_norm, t, a.hidden);
                }
                if (!(pieces >> piece & 1)) continue;
                if (piece == kStepAttend) {
                    if (has_attn) step_attend_stage(a, sh, rl, ly.q_norm != nullptr, kvh, split, kc, vc, tag, t, deadline);
                    step_head_weights(a, rl, next, t);
                    if (has_merge) step_merge(a, behind, tag, t, deadline);
                    continue;
                }
                const bool qkv = piece == kStepQkv, o = piece == kStepOut, gu = piece == kStepGateUp;
                const u32x4* row = qkv ? a.x : o ? a.attn : gu ? a.x2 : a.act;
                const uint32_t n = qkv || gu ? a.hidden : o ? qd : a.ffn;
                const f32x4 weights[2] = {qkv ? attn_w[0] : ffn_w[0], qkv ? attn_w[1] : ffn_w[1]};
                const auto stage = [&](auto rounds) {
                    step_stage<decltype(rounds)::value>(a, sh, sfrag, t, row, qkv ? x0 : nullptr, n, qkv || gu, weights, qkv ? tag - 1 : tag,
                                                        deadline, o ? a.x : qkv || gu ? nullptr : a.x2, o ? x0 : nullptr, o ? tag - 1 : tag, b);
                };
                if (n <= 1024)
                    stage(std::integral_constant<int, 1>());
                else if (n <= 2048)
                    stage(std::integral_constant<int, 2>());
                else
                    stage(std::integral_constant<int, 3>());
            }
        }
        return;
    }
    // What the staging waves poll for comes back behind all loads that the compute waves have made before: weights or
    // keys that are asked for while a row is on its way hold it up by their own trip (the Q/K/V row reached attention 1.8 to
    // 2.6 us after its last value was out; 1.1 to 1.6 now).  So a layer's first keys are asked for ahead of
    // its Q/K/V weights.
    StepLayer next = step_layer(a, 0);
    for (uint32_t L = 0; L < a.n_layers; L++) {
        const StepLayer ly = next;
        next = step_layer(a, min(L + 1, a.n_layers - 1));
        const uint32_t tag = a.tag0 + L;
        const uint16_t* kc = reinterpret_cast<const uint16_t*>(a.slab + 2 * L * a.side);
        const uint16_t* vc = reinterpret_cast<const uint16_t*>(a.slab + (2 * L + 1) * a.side);
        int ln = lane;
        const auto apart = [&] { asm volatile("" : "+v"(ln)); };     // what a piece derives from the lane is not kept through the others
        DecodeFrag<128> fa;
        if (has_attn) step_first_tile(a, fa, kvh, split, kc, vc, lane, wave);
        f32x4 acc[1], r, resid;
        float sc;
        if (has_qkv) {
            step_product<1>(sh, sfrag, acc, sc, resid, (StepWeights)ly.wqkv, b, b, a.hidden, true, ln, wave);
            if (wave == 0) {
#pragma unroll
                for (int i = 0; i < 4; i++) r[i] = acc[0][i] * sc;
                step_publish(a.qkv, width, 1, b, ln, r, tag);    // (a head's share is read by its own workgroups only)
            }
        }
        apart();
        if (has_attn) step_attend(a, sh, fa, kvh, split, kc, vc, tag, ln, wave);
        apart();
        if (has_o) {
            step_product<1>(sh, sfrag, acc, sc, resid, (StepWeights)ly.wo, b, b, qd, false, ln, wave);
            if (wave == 0) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float x = acc[0][i] * sc;
                    r[i] = x + resid[i];
                }
                step_publish(a.x2, a.hidden, kStepCopies, b, ln, r, tag);
            }
        }
        apart();
        if (has_gu) {
            f32x4 two[2], none;
            step_product<2>(sh, sfrag, two, sc, none, (StepWeights)ly.wgu, behind, behind + a.ffn / 16, a.hidden, true, ln, wave);
            if (wave == 0) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    float x = two[0][i] * sc, y = two[1][i] * sc;
                    asm volatile("" : "+v"(x), "+v"(y));     // the products end here: no contraction into the activation
                    r[i] = silu_mul(x, y);
                }
                step_publish(a.act, a.ffn, kStepCopies, behind, ln, r, tag);
            }
        }
        apart();
        if (has_o) {
            step_product<1>(sh, sfrag, acc, sc, resid, (StepWeights)ly.wdown, b, b, a.ffn, false, ln, wave);
            if (wave == 0) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float x = acc[0][i] * sc;
                    r[i] = x + resid[i];
                }
                if (L + 1 == a.n_layers) {
                    if ((ln & 15) == 0) *reinterpret_cast<f32x4*>(a.y + b * 16 + 4 * (ln >> 4)) = r;
                } else {
                    step_publish(a.x, a.hidden, kStepCopies, b, ln, r, tag);
                }
            }
        }
        apart();
    }
}

}  // namespace wr
