// C ABI of the MI355X attention path: device state, cache slabs, argument
// checking and kernel launches.  Declarations and the reference interfaces
// each entry point stands in for are in include/wr_hip_attn.h.
//
// There is no CPU path in this file: without a gfx950 device init fails and
// every other entry point returns WR_HIP_ERR_STATE.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <new>
#include <vector>

#include "../../include/wr_hip_attn.h"
#include "common.hip.h"
#include "runtime.hip.h"
#include "kernels_append.hip.h"
#include "kernels_decode.hip.h"
#include "kernels_prefill.hip.h"
#include "kernels_prefill_il.hip.h"
#include "kernels_prefill_pair.hip.h"
#include "kernels_prefill_ild.hip.h"
#include "prefill_plan.h"
#include "kernels_proj.hip.h"
#include "kernels_rows.hip.h"
#include "kernels_step.hip.h"
#include "step_gate.h"

using namespace wr;

// Scratch of wr_hip_attn_decode_batched_dev_noalloc, the one entry point that
// allocates nothing: the split-K tickets (first kNoAllocTicketBytes) and the
// partial rows (the rest).  Every device the library runs on holds its own copy
// until the process ends.  In host code the array's name is only a stand-in: the
// device address is asked for once per device at init (hipGetSymbolAddress) and
// kept in Lib::noalloc_ws; host code uses that pointer, never the name.
constexpr size_t kNoAllocTicketBytes = 64u * 1024u;            // 16 sessions x 1024 heads
constexpr size_t kNoAllocScratchBytes = 20u * 1024u * 1024u;   // tickets + partials
constexpr uint32_t kNoAllocMaxHeads = (uint32_t)(kNoAllocTicketBytes / sizeof(uint32_t) / WR_HIP_BATCH_MAX);
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

// Clears n 32-bit words (tickets).  A kernel rather than a memset call so that a
// caller may record the launch into a graph.
__global__ void fill_u32_kernel(uint32_t* p, uint32_t n, uint32_t v)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

struct wr_hip_weight {
    uint32_t n_out, n_in;
    void* tiles;                 // F16, tile order (kernels_proj.hip.h)
    size_t bytes;
};

struct wr_hip_kv {
    uint32_t n_layers, nkv, max_ctx, ctx_pad;
    uint32_t hd[WR_HIP_MAX_LAYERS];
    size_t k_off[WR_HIP_MAX_LAYERS];     // byte offsets into slab
    size_t vt_off[WR_HIP_MAX_LAYERS];
    uint8_t* slab;
    size_t bytes;
    int device;
    std::atomic<uint32_t> written{0};    // positions from here on have never been appended, in any layer

    void writes(uint64_t end)            // every call that appends says so
    {
        uint32_t w = written.load(std::memory_order_relaxed);
        while (w < end && !written.compare_exchange_weak(w, (uint32_t)end, std::memory_order_relaxed)) {}
    }
};

// What a model's steps in one launch keep: the layers' weights as the kernel reads them, and the rows that travel
// between its workgroups.  Used by one launch at a time (Lib::step_owner).
struct wr_hip_attn_step {
    uint32_t n_layers, hidden, ffn, nq, nkv;
    float eps;
    StepLayer* layers;                   // device
    u32x4* rows;                         // device: tagged rows, then partial rows
    size_t row_bytes;
    uint32_t next_tag;
};

namespace wr {

Lib g;
thread_local Ctx* cx = nullptr;

void logmsg(int level, const char* fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    if (g.log_fn)
        g.log_fn(level, buf, g.log_user);
    else
        fprintf(stderr, "[wr_hip_attn] %s\n", buf);
}

int hip_fail(hipError_t e, const char* what, uint32_t layer)
{
    logmsg(0, "hip: %s failed at layer %u: %s", what, layer, hipGetErrorString(e));
    return (e == hipErrorOutOfMemory) ? WR_HIP_ERR_NOMEM : WR_HIP_ERR_INTERNAL;
}

// Device memory of ended caches, for the next ones of their size: taking and giving back half a GiB is a third of a
// millisecond a session, and thousands of sessions one after the other come to minutes in which the driver, which
// clears what it is given back, takes 12 ms to each (a session of 10 tokens and one answer 2.1 -> 14.1 ms from some 250
// sessions on, with calls 2.1 ms apart; 400 at 2.6).  Bounded, the longest kept goes first; given back with
// the library, with a model (wr_hip_attn_trim), and when an allocation fails.  Nobody else's allocation can ask for it:
// where less than a sixteenth of the device is free nothing is kept.
constexpr size_t kKeptSlabs = 16, kKeptSlabBytes = (size_t)2 << 30;
constexpr size_t kKeptOfFree = 16;

void slabs_free(std::vector<Lib::Slab>& slabs)
{
    for (const Lib::Slab& s : slabs) (void)hipFree(s.p);
    slabs.clear();
}

// Everything kept: true if there was something.
bool slabs_trim()
{
    std::vector<Lib::Slab> out;
    {
        std::lock_guard<std::mutex> lk(g.slab_mu);
        out.swap(g.slabs);
    }
    const bool any = !out.empty();
    slabs_free(out);
    return any;
}

bool slab_take(size_t bytes, Lib::Slab& taken)
{
    std::lock_guard<std::mutex> lk(g.slab_mu);
    for (size_t i = 0; i < g.slabs.size(); i++)
        if (g.slabs[i].bytes == bytes) {
            taken = g.slabs[i];
            g.slabs.erase(g.slabs.begin() + (ptrdiff_t)i);
            return true;
        }
    return false;
}

// What the cache that had this memory left in it, cleared on the calling thread's stream: its own positions, not all that there is room for.
// A session's start behind one of 9 positions, of 28 layers of 8 heads of 128 with room for 4096: 60.3 us, now 5.8.  Past half of the room the
// fill of everything in one run takes less than the pieces would.
hipError_t slab_clear(const Lib::Slab& s)
{
    if (s.cleared.tiles == 0) return hipSuccess;
    if (s.cleared.tiles * 2 >= s.cleared.ctx_pad / kTileKeys || s.cleared.nkv > 0xFFFF / 2)   // (nearly all of it; no grid)
        return hipMemsetAsync(s.p, 0, s.bytes, cx->stream);
    // eight workgroups to a layer's head, and more where there are few of these: 2048 in all, of four stores a thread and more
    uint32_t hd = 0;
    for (uint32_t L = 0; L < s.n_layers; L++) hd = std::max(hd, s.cleared.hd[L]);
    const uint64_t stores = (uint64_t)s.cleared.tiles * kTileKeys * hd / 8, spread = 2048 / (2 * s.cleared.nkv * s.n_layers);
    const uint32_t x = (uint32_t)std::max<uint64_t>(8, std::min(spread, stores / 1024));
    hipLaunchKernelGGL(clear_cache_kernel, dim3(x, 2 * s.cleared.nkv, s.n_layers), dim3(256), 0, cx->stream, s.cleared, s.p);
    return hipGetLastError();
}

// The slab of a cache that has ended, on the library's device.  As hipFree would, it waits for all of the device's streams.
void slab_leave(const wr_hip_kv* kv)
{
    uint8_t* const p = kv->slab;
    const size_t bytes = kv->bytes;
    size_t free_bytes = 0, total = 0;
    const bool room = hipMemGetInfo(&free_bytes, &total) == hipSuccess && free_bytes >= total / kKeptOfFree;
    if (!room) (void)slabs_trim();
    if (!room || bytes > kKeptSlabBytes || hipDeviceSynchronize() != hipSuccess) {
        (void)hipGetLastError();
        (void)hipFree(p);
        return;
    }
    Lib::Slab s{};
    s.p = p;
    s.bytes = bytes;
    s.n_layers = kv->n_layers;
    s.cleared.nkv = kv->nkv;
    s.cleared.ctx_pad = kv->ctx_pad;
    s.cleared.tiles = (kv->written.load(std::memory_order_relaxed) + kTileKeys - 1) / kTileKeys;
    for (uint32_t L = 0; L < kv->n_layers; L++) {
        s.cleared.hd[L] = kv->hd[L];
        s.cleared.k_off[L] = kv->k_off[L];
        s.cleared.vt_off[L] = kv->vt_off[L];
    }
    std::vector<Lib::Slab> out;
    {
        std::lock_guard<std::mutex> lk(g.slab_mu);
        size_t kept = bytes;
        for (const Lib::Slab& s : g.slabs) kept += s.bytes;
        while (!g.slabs.empty() && (kept > kKeptSlabBytes || g.slabs.size() >= kKeptSlabs)) {
            kept -= g.slabs.front().bytes;
            out.push_back(g.slabs.front());
            g.slabs.erase(g.slabs.begin());
        }
        g.slabs.push_back(s);
    }
    slabs_free(out);
}

// For tests (wr_hip_attn_set_alloc_failures): true where an allocation is to fail, with a call's error left behind as a refused
// allocation leaves its own.
static bool alloc_refused()
{
    if (!g.fail_allocs.load(std::memory_order_relaxed) || count_down(g.fail_after) || !count_down(g.fail_allocs)) return false;
    (void)hipSetDevice(-1);
    return true;
}

// hipMalloc that what is kept makes room for.
hipError_t device_malloc(void** p, size_t bytes)
{
    const auto take = [&] { return alloc_refused() ? hipErrorOutOfMemory : hipMalloc(p, bytes); };
    hipError_t e = take();
    if (e != hipSuccess && slabs_trim()) {
        (void)hipGetLastError();
        e = take();
    }
    if (e != hipSuccess) (void)hipGetLastError();          // (the caller may do without: not for the next launch's check to find)
    return e;
}

// hipHostMalloc: no error of it is left behind either.
static hipError_t host_malloc(void** p, size_t bytes, unsigned flags = hipHostMallocDefault)
{
    const hipError_t e = alloc_refused() ? hipErrorOutOfMemory : hipHostMalloc(p, bytes, flags);
    if (e != hipSuccess) (void)hipGetLastError();
    return e;
}

int ensure_device(Buffer& b, size_t need)
{
    if (need <= b.cap) return WR_HIP_OK;
    HIP_TRY(hipStreamSynchronize(cx->stream), "sync before workspace growth", 0);
    if (b.p) (void)hipFree(b.p);
    b.p = nullptr;
    b.cap = 0;
    const size_t want = need + need / 2 + 4096;
    HIP_TRY(device_malloc(&b.p, want), "workspace alloc", 0);
    b.cap = want;
    return WR_HIP_OK;
}

// The same for memory that a launch can do without, in a buffer of its own: nothing another launch must have
// is given up to make it, and a refusal is no error.  A power of two of MiB; the old one goes only when the new one is
// there.  False: there is none, and the launch does without (as do the next ones: asking costs a failed call each time).
bool optional_device(Buffer& b, uint32_t& refused, size_t need, const char* without)
{
    if (need <= b.cap) return true;
    if (refused) {
        refused--;
        return false;
    }
    size_t want = (size_t)1 << 20;
    while (want < need) want *= 2;
    void* bigger = nullptr;
    if (device_malloc(&bigger, want) != hipSuccess) {
        logmsg(1, "no %zu MiB for %s", want >> 20, without);
        refused = kRefusedLaunches;
        return false;
    }
    if (b.p) {                                     // launches that use it may still be on their way
        if (hipStreamSynchronize(cx->stream) != hipSuccess) {
            (void)hipFree(bigger);
            return false;
        }
        (void)hipFree(b.p);
    }
    b.p = bigger;
    b.cap = want;
    return true;
}

int ensure_pinned(Buffer& b, size_t need)
{
    if (need <= b.cap) return WR_HIP_OK;
    HIP_TRY(hipStreamSynchronize(cx->stream), "sync before pinned growth", 0);
    if (b.p) (void)hipHostFree(b.p);
    b.p = nullptr;
    b.cap = 0;
    const size_t want = need + need / 2 + 4096;
    HIP_TRY(host_malloc(&b.p, want), "pinned alloc", 0);
    b.cap = want;
    return WR_HIP_OK;
}

// Puts the split-K tickets back to zero.  They return to zero by themselves at
// the end of every launch that completes; after a launch or a wait has failed
// nothing is known about them, and a non-zero ticket would make the next launch
// merge partial rows that were never written.
void reset_tickets()
{
    if (!cx->d_counters) return;
    const size_t cb = (size_t)WR_HIP_BATCH_MAX * kMaxHeads * sizeof(uint32_t);
    if (hipMemsetAsync(cx->d_counters, 0, cb, cx->stream) == hipSuccess) (void)hipStreamSynchronize(cx->stream);
    (void)hipGetLastError();
}

// Waits for the calling thread's stream, then looks at the error word.  Every entry point
// that promises results on return waits through here, so a kernel that gave up a
// bounded wait (and went on with wrong data) turns into WR_HIP_ERR_INTERNAL on the
// first call that could hand those results to the caller, logged with the layer
// (as the reference reports op failures, src/core/session.c:170-174).
int sync_checked(const char* what, uint32_t layer)
{
    const hipError_t e = hipStreamSynchronize(cx->stream);
    if (e != hipSuccess) {
        const int rc = hip_fail(e, what, layer);
        reset_tickets();
        return rc;
    }
    const uint32_t w = cx->err_host ? *cx->err_host : 0u;
    if (w != 0) {
        *cx->err_host = 0;
        logmsg(0, "device: a kernel's bounded wait expired at layer %u (error word 0x%08x, seen at: %s); "
                  "results produced since the previous wait are invalid", w & kDevErrLayerMask, w, what);
        reset_tickets();
        return WR_HIP_ERR_INTERNAL;
    }
    return WR_HIP_OK;
}

// Host -> device / device -> host on the stream.  Small transfers go
// through pinned staging (predictable latency); large ones are handed to the
// runtime directly.  Both leave the stream synchronised for the host buffer.
int copy_up(void* dst_dev, const void* src_host, size_t bytes, size_t pin_off)
{
    if (bytes == 0) return WR_HIP_OK;
    if (pin_off + bytes <= cx->h_pin.cap && bytes <= kPinSmall) {
        memcpy((uint8_t*)cx->h_pin.p + pin_off, src_host, bytes);
        HIP_TRY(hipMemcpyAsync(dst_dev, (uint8_t*)cx->h_pin.p + pin_off, bytes,
                               hipMemcpyHostToDevice, cx->stream), "h2d", 0);
    } else {
        HIP_TRY(hipMemcpyAsync(dst_dev, src_host, bytes, hipMemcpyHostToDevice, cx->stream),
                "h2d", 0);
        HIP_TRY(hipStreamSynchronize(cx->stream), "h2d sync", 0);
    }
    return WR_HIP_OK;
}

int copy_down_sync(void* dst_host, const void* src_dev, size_t bytes)
{
    if (bytes == 0) return sync_checked("sync", 0);
    if (bytes <= cx->h_pin.cap && bytes <= kPinSmall) {
        HIP_TRY(hipMemcpyAsync(cx->h_pin.p, src_dev, bytes, hipMemcpyDeviceToHost, cx->stream),
                "d2h", 0);
        int rc = sync_checked("d2h sync", 0);
        if (rc) return rc;
        memcpy(dst_host, cx->h_pin.p, bytes);
    } else {
        HIP_TRY(hipMemcpyAsync(dst_host, src_dev, bytes, hipMemcpyDeviceToHost, cx->stream),
                "d2h", 0);
        int rc = sync_checked("d2h sync", 0);
        if (rc) return rc;
    }
    return WR_HIP_OK;
}

}  // namespace wr

namespace {

bool mfma_shape(uint32_t hd, uint32_t group)
{
    return !g.force_generic && (hd == 64 || hd == 128 || hd == 256) && group <= kMaxGroupMfma;
}

int check_layer(const wr_hip_kv* kv, uint32_t layer)
{
    if (!kv) return WR_HIP_ERR_INVAL;
    if (layer >= kv->n_layers || kv->hd[layer] == 0) return WR_HIP_ERR_INVAL;
    return WR_HIP_OK;
}

uint32_t key_lo_for(uint32_t window, uint32_t seq_k)
{
    return (window > 0 && seq_k > window) ? seq_k - window : 0;
}

// ------------------------------------------------------------------------
// Bodies (the caller has entered: device current, cx set).

template <typename Src>
int append_rows_locked(wr_hip_kv* kv, uint32_t layer, uint32_t pos, uint32_t n_rows,
                       const Src* k_dev, const Src* v_dev)
{
    const uint32_t hd = kv->hd[layer], nkv = kv->nkv;
    kv->writes((uint64_t)pos + n_rows);
    uint16_t* kbase = reinterpret_cast<uint16_t*>(kv->slab + kv->k_off[layer]);
    uint16_t* vbase = reinterpret_cast<uint16_t*>(kv->slab + kv->vt_off[layer]);
    const uint32_t nblk = (pos + n_rows - 1) / kVBlock - pos / kVBlock + 1;
    const uint32_t runs = (hd + kAppendDims - 1) / kAppendDims;
    // vectors of eight dimensions: where they are whole and the sources lie on 16 bytes (and the grid's second
    // dimension has room for the heads)
    if (hd % 8 == 0 && (((uintptr_t)k_dev | (uintptr_t)v_dev) & 15) == 0 && (uint64_t)nkv * runs < 65536) {
        hipLaunchKernelGGL(HIP_KERNEL_NAME(append_kv_kernel<Src>), dim3(nblk, nkv * runs, 2), dim3(256), 0, cx->stream,
                           k_dev, v_dev, kbase, vbase, pos, n_rows, nkv, hd, kv->ctx_pad);
        HIP_TRY(hipGetLastError(), "append launch", layer);
        return WR_HIP_OK;
    }
    const size_t total = (size_t)n_rows * nkv * hd;
    const uint32_t blocks = (uint32_t)((total + 255) / 256);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(append_k_kernel<Src>), dim3(blocks), dim3(256), 0, cx->stream,
                       k_dev, kbase, pos, n_rows, nkv, hd, kv->ctx_pad);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(append_v_kernel<Src>), dim3((hd + 63) / 64, nkv, nblk),
                       dim3(256), 0, cx->stream, v_dev, vbase, pos, n_rows, nkv, hd, kv->ctx_pad);
    HIP_TRY(hipGetLastError(), "append launch", layer);
    return WR_HIP_OK;
}

int check_append(const wr_hip_kv* kv, uint32_t layer, uint32_t pos, uint32_t n_rows,
                 const void* k, const void* v)
{
    if (!g.inited) return WR_HIP_ERR_STATE;
    int rc = check_layer(kv, layer);
    if (rc) return rc;
    if (n_rows == 0) return WR_HIP_OK;
    if (!k || !v) return WR_HIP_ERR_INVAL;
    if ((uint64_t)pos + n_rows > kv->max_ctx) return WR_HIP_ERR_CTX_FULL;
    return WR_HIP_OK;
}

// Where a launch keeps its split-K tickets and partial rows: the library's own
// growable buffers (ws == nullptr), or a fixed workspace that is never grown.
struct DecodeWorkspace {
    unsigned char* ws = nullptr;     // tickets at 0, partials from ticket_bytes on
    size_t ticket_bytes = 0;
    size_t bytes = 0;
};

struct SplitRule {
    uint32_t tiles_per_wg, tail, n_splits;
    bool pairs, shorts;      // long and short sessions, whose splits may share a workgroup
};

// The rule looks at ONE session only (its own visible
// key range), never at the rest of the batch: a session's arithmetic is then
// the same whether it is stepped alone or with others, which is what makes
// the batched step bit-identical to serial steps (reference contract:
// src/core/batch.c:15-19).  Half a MiB of K+V per workgroup (1024 keys at
// head_dim 128, 512 at 256): 16 sessions of 4096 run as fast with it as
// with twice that, and a single session's chain of tiles is half as long
// (one session of 8192 keys: 27 -> 17 us); from
// 8K keys up an eighth of the session per workgroup measured better
// (fewer partials and workgroup turnovers: 82 % -> 86 % of HBM peak at
// 16 x 32768).  A short session (up to 2048 keys at head_dim 128) takes a
// quarter of that per workgroup: its launch is a chain of latencies, and a
// workgroup that has all its tiles in flight at once ends sooner than one
// that walks eight of them per wave (one session of 1024 keys: 12.0 -> 7.8 us,
// of 2048: 13.8 -> 8.2 us; 16 sessions of ~520: the step of a 28-layer model
// 2.03 -> 1.89 ms).  A medium session (more than 2048 and fewer than 4096 keys)
// takes half: one session of 3000 keys 14 -> 10.6 us, the ragged batch of 16
// 35.2 -> 34.6 us; at 4096 keys and beyond the full figure stands (16 x 4096
// loses 4-8 % with halves).  The session's tiles are spread evenly over the workgroups,
// and the floor keeps the in-kernel merge within kMaxSplits partials.
// A long session (from 8K keys up at head_dim 128) is cut into twice as
// many splits as it gets workgroups in a full launch, and a workgroup there
// works through two consecutive splits, one after the other: the unit of
// arithmetic (a split: one partial, the tiles dealt to the four waves in
// turn) stays a function of the session alone, while a launch too small to
// give every CU a workgroup sends each split to a workgroup of its own.
// One session of 8192 keys: 64 -> 128 workgroups, 14.8 -> 11.2 us; of 16384:
// 24.5 -> 16.2; of 32768: 43.9 -> 26.9.  The price in a full launch is one
// extra merge of the four waves per workgroup: not measurable at 16 x 32768.
// (The same from 4096 keys up costs 16 x 4096 4.5 %: those workgroups have
// 32 tiles, and the waves meeting in the middle is 2 us of their 40.)
// A caller that serves one session at a time can go further with
// wr_hip_attn_set_tuning.
SplitRule split_rule(uint32_t tiles, uint32_t hd, bool use_mfma, uint32_t tune)
{
    SplitRule r{};
    uint32_t tpw, tail = 0;
    if (tune) {
        tpw = tune / kTileKeys;
        if (tpw == 0) tpw = 1;
    } else {
        uint32_t cap = kDefaultTilesPerWg * 128u / (hd < 32 ? 32 : hd);
        if (cap == 0) cap = 1;
        if (tiles <= 2 * cap) {                                  // a short session: see above
            cap = cap >= 4 ? cap / 4 : 1;
            // ... whose LAST four tiles are a split of their own: one tile per
            // wave.  In a decode step the last tile holds the new position: the
            // workgroup that has it also makes the new row's K and V and patches
            // them in, and with a full share of tiles on top it finishes last and
            // the merge waits for it (timestamps: its ticket 2 us after the
            // others').  With one tile per wave it finishes first, and a workgroup
            // that is done anyway merges: the decode step of a 28-layer model at
            // ~520 keys 1.02 -> 1.00 ms, sixteen sessions 1.90 -> 1.87 ms.  (A tail
            // of ONE tile does the same for one session and costs sixteen 2-3 %:
            // it adds a workgroup per session and KV head.)  A caller that has
            // appended the row itself pays for the extra split instead: one
            // session of 1024 keys 7.8 -> 8.2 us, of 2048 keys 8.1 -> 8.8 us.
            if (tiles >= 6) tail = 4;
            // In a launch that would not find a place for every split at once two
            // consecutive splits of a short session share a workgroup as well (the
            // splits keep their size): see below.
            r.shorts = use_mfma && hd <= 128;
        } else if (tiles < 4 * cap) {
            cap = cap >= 2 ? cap / 2 : 1;                           // a medium one: see above
        } else if (cap <= tiles / 8) {
            cap = tiles / 8;
            r.pairs = use_mfma && hd <= 128;                       // a long one: see above
        }
        const uint32_t body = tiles - tail;
        const uint32_t want = (body + cap - 1) / cap;              // workgroups
        tpw = (body + want - 1) / want;                            // even share
        if (r.pairs) tpw = (tpw + 1) / 2;                         // two splits per workgroup
        if (r.shorts) r.pairs = true;
    }
    const uint32_t body = tiles - tail;
    const uint32_t room = kMaxSplits - (tail ? 1u : 0u);
    const uint32_t floor_tiles = (body + room - 1) / room;
    if (tpw < floor_tiles) tpw = floor_tiles;
    r.tiles_per_wg = tpw;
    r.tail = tail;
    r.n_splits = (body + tpw - 1) / tpw + (tail ? 1u : 0u);
    return r;
}

int decode_locked(uint32_t n, wr_hip_kv* const* kv, uint32_t layer, const uint32_t* seq_k,
                  const float* q_dev, float* out_dev, uint32_t nq, float scale_override,
                  uint32_t window, const DecodeWorkspace& fixed = DecodeWorkspace(),
                  const DecodeFusedArgs* fused = nullptr)
{
    const uint32_t hd = kv[0]->hd[layer], nkv = kv[0]->nkv;
    const uint32_t group = nq / nkv;
    const bool use_mfma = mfma_shape(hd, group);

    DecodeArgs a;
    memset(&a, 0, sizeof a);
    uint32_t tiles[kBatchMax];
    for (uint32_t i = 0; i < n; i++) {
        DecodeSession& s = a.s[i];
        s.k = reinterpret_cast<const uint16_t*>(kv[i]->slab + kv[i]->k_off[layer]);
        s.vt = reinterpret_cast<const uint16_t*>(kv[i]->slab + kv[i]->vt_off[layer]);
        s.seq_k = seq_k[i];
        s.key_lo = key_lo_for(window, seq_k[i]);
        s.ctx_pad = kv[i]->ctx_pad;
        tiles[i] = (s.seq_k + kTileKeys - 1) / kTileKeys - s.key_lo / kTileKeys;
    }

    uint32_t max_splits = 1;
    const uint32_t tune = g.tune_keys_per_wg.load(std::memory_order_relaxed);
    bool pairs[kBatchMax], shorts[kBatchMax];
    uint32_t wgs_paired = 0, wgs_shorts_alone = 0;
    for (uint32_t i = 0; i < n; i++) {
        const SplitRule r = split_rule(tiles[i], hd, use_mfma, tune);
        pairs[i] = r.pairs;
        shorts[i] = r.shorts;
        a.s[i].tiles_per_wg = r.tiles_per_wg;
        a.s[i].tail_tiles = (uint16_t)r.tail;
        a.s[i].parts_per_wg = 1;
        a.s[i].n_splits = r.n_splits;
        if (a.s[i].n_splits > max_splits) max_splits = a.s[i].n_splits;
        const uint32_t halves = (a.s[i].n_splits + 1) / 2;
        wgs_paired += pairs[i] ? halves : a.s[i].n_splits;
        wgs_shorts_alone += pairs[i] && !shorts[i] ? halves : a.s[i].n_splits;
    }
    // The launch as a whole decides this, not the session: it changes which
    // workgroup does a split, never the split.  Splits of short sessions keep a
    // workgroup each as long as all of the launch's workgroups run at once (three per
    // CU): a split alone has its tiles in flight from the start and one merge behind
    // them, and half the places standing empty is the larger loss (sixteen sessions of
    // 100 .. 1500 keys, 36 entries against 65 per KV head: 18.0 -> 16.8 us; the ragged
    // batch of 16, 736 workgroups, 27.6 -> 26.8).  Beyond that a second round of
    // workgroups costs more than the pairing (a batch of 816 entries: 33.5 us alone,
    // 32.8 paired).
    const bool shorts_pair = (uint64_t)wgs_shorts_alone * nkv > (uint64_t)g.n_cus * 3;
    if ((uint64_t)wgs_paired * nkv >= g.n_cus)
        for (uint32_t i = 0; i < n; i++)
            if (pairs[i] && (!shorts[i] || shorts_pair)) a.s[i].parts_per_wg = 2;
    // work list, longest entries first (ties keep session, split order)
    {
        uint32_t len[kBatchMax * kMaxSplits];
        uint32_t cnt = 0;
        for (uint32_t i = 0; i < n; i++) {
            const uint32_t body = tiles[i] - a.s[i].tail_tiles;
            const uint32_t ppw = a.s[i].parts_per_wg;
            for (uint32_t wg = 0; wg * ppw < a.s[i].n_splits; wg++) {
                uint32_t l = 0;
                for (uint32_t sp = wg * ppw; sp < (wg + 1) * ppw && sp < a.s[i].n_splits; sp++) {
                    if (a.s[i].tail_tiles && sp == a.s[i].n_splits - 1) {
                        l += a.s[i].tail_tiles;
                    } else {
                        const uint32_t begin = sp * a.s[i].tiles_per_wg;
                        const uint32_t left = body - begin;
                        l += left < a.s[i].tiles_per_wg ? left : a.s[i].tiles_per_wg;
                    }
                }
                len[cnt] = l;
                a.items[cnt++] = (uint16_t)((i << 8) | wg);
            }
        }
        for (uint32_t i = 1; i < cnt; i++) {           // insertion sort: at most 1024 entries
            const uint32_t l = len[i];
            const uint16_t it = a.items[i];
            uint32_t j = i;
            while (j > 0 && len[j - 1] < l) {
                len[j] = len[j - 1];
                a.items[j] = a.items[j - 1];
                j--;
            }
            len[j] = l;
            a.items[j] = it;
        }
        a.n_items = cnt;
    }
    a.q = q_dev;
    a.out = out_dev;
    a.nq = nq;
    a.nkv = nkv;
    a.group = group;
    a.hd = hd;
    a.max_splits = max_splits;
    a.counters = fixed.ws ? reinterpret_cast<uint32_t*>(fixed.ws) : cx->d_counters;
    const float scale = (scale_override > 0.0f) ? scale_override : 1.0f / sqrtf((float)hd);
    a.qscale = scale * kLog2e;

    if (max_splits > 1) {
        const size_t po = (size_t)n * nq * max_splits * hd * sizeof(float);
        const size_t pml = (size_t)n * nq * max_splits * 2 * sizeof(float);
        uint8_t* base;
        if (fixed.ws) {
            if (fixed.ticket_bytes + po + pml > fixed.bytes) {
                logmsg(0, "decode (no-alloc form): %zu bytes of split-K partials exceed the fixed "
                          "workspace of %zu bytes (layer %u)", po + pml, fixed.bytes - fixed.ticket_bytes,
                       layer);
                return WR_HIP_ERR_LIMIT;
            }
            base = fixed.ws + fixed.ticket_bytes;
        } else {
            int rc = ensure_device(cx->d_part, po + pml);
            if (rc) return rc;
            base = reinterpret_cast<uint8_t*>(cx->d_part.p);
        }
        a.part_o = reinterpret_cast<float*>(base);
        a.part_ml = reinterpret_cast<float*>(base + po);
        if (fixed.ws) {
            // the array keeps the last call's contents: the tickets this launch
            // uses must start at zero
            const uint32_t words = n * (use_mfma ? nkv : nq);
            hipLaunchKernelGGL(fill_u32_kernel, dim3((words + 255) / 256), dim3(256), 0, cx->stream,
                               a.counters, words, 0u);
        }
    }

    if (fused && !(use_mfma && hd == 128)) return WR_HIP_ERR_UNSUPPORTED;
    if (fused)
        for (uint32_t i = 0; i < n; i++) kv[i]->writes(seq_k[i]);
    if (use_mfma) {
        const dim3 grid(nkv, a.n_items), block(kDecodeThreads);
        DecodeFusedArgs none;
        memset(&none, 0, sizeof none);
        if (fused)
            launch_main(decode_mfma_kernel<128, true>, grid, block, a, *fused, 0);
        else if (hd == 64)
            launch_main(decode_mfma_kernel<64>, grid, block, a, none, 0);
        else if (hd == 128)
            launch_main(decode_mfma_kernel<128>, grid, block, a, none, 0);
        else
            launch_main(decode_mfma_kernel<256>, grid, block, a, none, 0);
    } else {
        launch_main(decode_generic_kernel, dim3(nq, a.n_items), dim3(kDecodeThreads), a);
    }
    {
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) {
            const int rc = hip_fail(e, "decode launch", layer);
            reset_tickets();
            return rc;
        }
    }
    return WR_HIP_OK;
}

int check_decode(uint32_t n, wr_hip_kv* const* kv, uint32_t layer, const uint32_t* seq_k,
                 const void* q, const void* out, uint32_t nq)
{
    if (!g.inited) return WR_HIP_ERR_STATE;
    if (!kv || !seq_k || !q || !out) return WR_HIP_ERR_INVAL;
    if (n == 0 || n > WR_HIP_BATCH_MAX) return WR_HIP_ERR_LIMIT;
    for (uint32_t i = 0; i < n; i++)
        if (!kv[i]) return WR_HIP_ERR_INVAL;
    // The reference counts an attention call once its pointer checks have passed
    // and before it looks at any shape (src/core/kernels.c:1418-1423), so calls
    // refused for their shapes count too: one per session here.
    g.calls.fetch_add(n, std::memory_order_relaxed);
    for (uint32_t i = 0; i < n; i++) {
        int rc = check_layer(kv[i], layer);
        if (rc) return rc;
        if (kv[i]->nkv != kv[0]->nkv || kv[i]->hd[layer] != kv[0]->hd[layer])
            return WR_HIP_ERR_INVAL;
        for (uint32_t j = 0; j < i; j++)
            if (kv[i] == kv[j]) return WR_HIP_ERR_INVAL;
    }
    if (nq == 0 || nq % kv[0]->nkv != 0) return WR_HIP_ERR_INVAL;
    if (nq > kMaxHeads) return WR_HIP_ERR_LIMIT;
    for (uint32_t i = 0; i < n; i++) {
        if (seq_k[i] == 0) return WR_HIP_ERR_INVAL;
        if (seq_k[i] > WR_HIP_ATTN_MAX_SEQ) return WR_HIP_ERR_LIMIT;
        if (seq_k[i] > kv[i]->max_ctx) return WR_HIP_ERR_INVAL;
    }
    return WR_HIP_OK;
}

// Room for the parts' rows, in a buffer of their own.  False: there is none, and the launch goes uncut.
bool prefill_parts_ready(PrefillArgs& a, uint32_t parts)
{
    const size_t rows = (size_t)parts * a.T * a.nq, o = rows * a.hd * sizeof(float), need = o + rows * 2 * sizeof(float);
    if (!optional_device(cx->d_prefill, cx->prefill_refused, need, "parts of long blocks; they go uncut")) return false;
    a.n_parts = parts;
    a.part_o = reinterpret_cast<float*>(cx->d_prefill.p);
    a.part_ml = reinterpret_cast<float*>(reinterpret_cast<uint8_t*>(cx->d_prefill.p) + o);
    return true;
}

int prefill_locked(wr_hip_kv* kv, uint32_t layer, uint32_t p0, uint32_t T, const float* q_dev,
                   float* out_dev, uint32_t nq, float scale_override, uint32_t window,
                   const uint16_t* q16_dev = nullptr)
{
    const uint32_t hd = kv->hd[layer];
    PrefillArgs a;
    memset(&a, 0, sizeof a);
    a.k = reinterpret_cast<const uint16_t*>(kv->slab + kv->k_off[layer]);
    a.vt = reinterpret_cast<const uint16_t*>(kv->slab + kv->vt_off[layer]);
    a.q = q_dev;
    a.q16 = q16_dev;
    a.out = out_dev;
    a.p0 = p0;
    a.T = T;
    a.nq = nq;
    a.nkv = kv->nkv;
    a.group = nq / kv->nkv;
    a.hd = hd;
    a.ctx_pad = kv->ctx_pad;
    a.window = window;
    const float scale = (scale_override > 0.0f) ? scale_override : 1.0f / sqrtf((float)hd);
    a.qscale = scale * kLog2e;
    const uint32_t G = a.group;
    const bool mfma = !g.force_generic && (hd == 64 || hd == 128 || hd == 256) &&
                      (G == 1 || G == 2 || G == 4 || G == 8);
    if (q16_dev && !(mfma && (hd == 64 || hd == 128))) return WR_HIP_ERR_UNSUPPORTED;
    if (mfma) {
        const bool one_wave = hd == 128 && !g.prefill_two_waves, four_waves = hd == 256 && g.prefill_256_four_waves;
        const PrefillSizes sizes = {p0, T, window, nq, kv->nkv, hd};
        const auto plan = [&](uint32_t parts) {
            return prefill_plan(sizes, g.n_cus, !one_wave && !four_waves, parts, (uint64_t)g.prefill_part_mb.load(std::memory_order_relaxed) << 20);
        };
        PrefillPlan p = plan(kMaxPrefillParts);
        if (p.parts > 1 && !prefill_parts_ready(a, p.parts)) p = plan(1);
        a.single = p.single;
        const dim3 grid(p.ny, p.single ? p.nblk : (p.nblk + 1) / 2, p.parts);
        if (one_wave) {
            if (q16_dev)
                launch_main(prefill_pair_kernel<128, true>, grid, dim3(kPairThreads), a, pair_smem_bytes<128>());
            else
                launch_main(prefill_pair_kernel<128, false>, grid, dim3(kPairThreads), a, pair_smem_bytes<128>());
        } else if (four_waves) {   // the earlier form: one wave per SIMD owns all 256 dimensions of its rows
            launch_main(prefill_mfma_kernel<256>, dim3(grid.y, grid.x), dim3(kPrefillThreads), a);
        } else {
            const auto launch = [&](auto np, auto part) {
                constexpr int NP = decltype(np)::value;
                constexpr bool PART = decltype(part)::value;
                if (hd == 64)
                    launch_main(prefill_il_kernel<64, NP, PART>, grid, dim3(split_threads(NP)), a, split_smem_bytes<64, NP>());
                else if (hd == 128)
                    launch_main(prefill_il_kernel<128, NP, PART>, grid, dim3(split_threads(NP)), a, split_smem_bytes<128, NP>());
                else   // 256: the wave sets divide the dimensions
                    launch_main(prefill_ild_kernel<NP, PART>, grid, dim3(split_threads(NP)), a, ild_smem_bytes<NP>());
            };
            const auto whole_or_parts = [&](auto np) {
                if (p.parts > 1)
                    launch(np, std::true_type());
                else
                    launch(np, std::false_type());
            };
            if (p.np == 2)
                whole_or_parts(std::integral_constant<int, 2>());
            else
                whole_or_parts(std::integral_constant<int, 4>());
            if (p.parts > 1) {
                HIP_TRY(hipGetLastError(), "prefill launch", layer);
                const uint32_t units = T * nq * (hd / 4);     // (bounded: few workgroups made these rows)
                hipLaunchKernelGGL(prefill_combine_kernel, dim3((units + 255) / 256), dim3(256), 0, cx->stream, a);
            }
        }
    } else {
        launch_main(prefill_generic_kernel, dim3(T, nq), dim3(kDecodeThreads), a);
    }
    HIP_TRY(hipGetLastError(), "prefill launch", layer);
    return WR_HIP_OK;
}

int check_prefill(const wr_hip_kv* kv, uint32_t layer, uint32_t p0, uint32_t T, const void* q,
                  const void* out, uint32_t nq)
{
    if (!g.inited) return WR_HIP_ERR_STATE;
    if (!kv || !q || !out) return WR_HIP_ERR_INVAL;
    // one count per row: prefill stands for T attention calls of the reference,
    // each counted after its pointer checks and before its shape checks
    // (src/core/kernels.c:1418-1423)
    g.calls.fetch_add(T, std::memory_order_relaxed);
    int rc = check_layer(kv, layer);
    if (rc) return rc;
    if (T == 0) return WR_HIP_ERR_INVAL;
    if (nq == 0 || nq % kv->nkv != 0) return WR_HIP_ERR_INVAL;
    if ((uint64_t)p0 + T > WR_HIP_ATTN_MAX_SEQ) return WR_HIP_ERR_LIMIT;
    if ((uint64_t)p0 + T > kv->max_ctx) return WR_HIP_ERR_INVAL;
    return WR_HIP_OK;
}

// ---- thread contexts -------------------------------------------------------

void ctx_destroy(Ctx* c)
{
    if (!c) return;
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    for (hipEvent_t e : c->ev) (void)hipEventDestroy(e);
    if (c->d_stage.p) (void)hipFree(c->d_stage.p);
    if (c->d_part.p) (void)hipFree(c->d_part.p);
    if (c->d_picked.p) (void)hipFree(c->d_picked.p);
    if (c->d_prefill.p) (void)hipFree(c->d_prefill.p);
    if (c->d_proj.p) (void)hipFree(c->d_proj.p);
    if (c->d_counters) (void)hipFree(c->d_counters);
    if (c->h_pin.p) (void)hipHostFree(c->h_pin.p);
    if (c->err_host) (void)hipHostFree((void*)c->err_host);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
}

// A new context: stream (default priority), staging, zeroed tickets, error word.
// Caller holds g.mu and has set the device.
Ctx* ctx_create()
{
    Ctx* c = new (std::nothrow) Ctx();
    if (!c) return nullptr;
    Ctx* const saved = cx;
    cx = c;                                  // the helpers below work on the current context
    int rc = WR_HIP_OK;
    hipError_t e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
    if (e != hipSuccess) rc = hip_fail(e, "stream create", 0);
    if (rc == WR_HIP_OK) rc = ensure_pinned(c->h_pin, 2 * kPinSmall);
    if (rc == WR_HIP_OK) rc = ensure_device(c->d_stage, 2 * kPinSmall);
    if (rc == WR_HIP_OK) {
        const size_t cb = (size_t)WR_HIP_BATCH_MAX * kMaxHeads * sizeof(uint32_t);
        e = device_malloc((void**)&c->d_counters, cb);
        if (e == hipSuccess) e = hipMemsetAsync(c->d_counters, 0, cb, c->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
        if (e != hipSuccess) rc = hip_fail(e, "ticket array", 0);
    }
    if (rc == WR_HIP_OK) {
        void* hp = nullptr;
        void* dp = nullptr;
        e = host_malloc(&hp, 64, hipHostMallocMapped);
        if (e == hipSuccess) e = hipHostGetDevicePointer(&dp, hp, 0);
        if (e != hipSuccess) {
            rc = hip_fail(e, "error word", 0);
            if (hp) (void)hipHostFree(hp);
        } else {
            memset(hp, 0, 64);
            c->err_host = reinterpret_cast<volatile uint32_t*>(hp);
            c->err_dev = reinterpret_cast<uint32_t*>(dp);
        }
    }
    cx = saved;
    if (rc != WR_HIP_OK) {
        ctx_destroy(c);
        return nullptr;
    }
    return c;
}

// Hands a thread's context back when the thread ends, for the next new thread
// (threads of a pool come and go; their streams and staging need not).
struct ThreadSlot {
    Ctx* c = nullptr;
    uint64_t generation = 0;
    ~ThreadSlot()
    {
        if (!c) return;
        std::lock_guard<std::mutex> lk(g.mu);
        if (g.inited && generation == g.generation) g.idle.push_back(c);
    }
};
thread_local ThreadSlot t_slot;

}  // namespace

namespace wr {

Entered::Entered()
{
    if (!g.inited) return;
    (void)hipSetDevice(g.device);
    if (!t_slot.c || t_slot.generation != g.generation) {
        std::lock_guard<std::mutex> lk(g.mu);
        if (!g.inited) return;
        Ctx* c = nullptr;
        if (!g.idle.empty()) {
            c = g.idle.back();
            g.idle.pop_back();
            c->profiling = false;            // the thread that had it before may have ended mid-measurement
            c->ev_used = 0;
            c->rows = 0;
        } else {
            c = ctx_create();
            if (c) g.ctxs.push_back(c);
        }
        t_slot.c = c;
        t_slot.generation = g.generation;
    }
    cx = t_slot.c;
    good = cx != nullptr;
    if (good) cx->depth.store(cx->depth.load(std::memory_order_relaxed) + 1, std::memory_order_relaxed);
}

}  // namespace wr
// projections: launch helpers (the caller has entered)
namespace {

template <int GROUPS, int NT, bool GATED = false>
void launch_proj(const ProjArgs& a)
{
    const uint32_t runs = (a.N / 16 + NT - 1) / NT;              // runs of 16*NT outputs
    const uint32_t per_block = 4 / a.ksplit;
    launch_main(proj_rows_kernel<GROUPS, NT, GATED>, dim3((runs + per_block - 1) / per_block), dim3(kProjThreads), a);
}

// Prefill-sized row counts: the largest tile that still fills the chip.
//   LDS-staged, eight waves, 256 outputs x 128 rows per workgroup, from one workgroup per CU;
//   LDS-staged, 128 x 128, from two workgroups per CU;
//   LDS-staged, 128 x 64, from one per CU (software-pipelined: a SIMD may hold a single wave);
//   registers, the four waves split the input range: 16 x 8 to 64 x 32.
constexpr int kProjGemmMinRows = 17;
constexpr uint32_t kProjGroupRows = 257;           // from here on the fragments are made by row groups: at 200 rows a
                                                   // workgroup per row is 0.6 to 2.2 us faster, at 300 as fast, at 511 1 us slower
constexpr size_t kProjRow1MaxLds = 60 * 1024;      // inputs up to 15 360 take the one-row kernel
static_assert(kProjRow1MaxLds + row1_static_lds(false) <= 64 * 1024, "what a kernel may use without asking");
static_assert(kProjRow1MaxLds + row1_static_lds(true) <= 160 * 1024, "gated: asked for at init");

template <int GROUPS, int NT, int D, bool GATED = false>
void launch_proj_gemm_split(const ProjArgs& a, uint32_t groups)
{
    launch_main(proj_gemm_split_kernel<GROUPS, NT, D, GATED>,
                dim3((a.N / 16 + NT - 1) / NT, (groups + GROUPS - 1) / GROUPS), dim3(kProjThreads), a);
}

// `per_xcd`: workgroups an XCD holds at once
template <int GROUPS, int WN, int RING, bool PIPE, int KS>
void launch_proj_lds(ProjArgs a, uint32_t groups, uint32_t per_xcd)
{
    uint32_t blocks = 0;
    a.cols = (uint8_t)xcd_cols((a.N / 16 + WN * 4 - 1) / (WN * 4), (groups + 2 * GROUPS - 1) / (2 * GROUPS), (uint64_t)a.N * a.K * 2,
                      (uint64_t)groups * 8 * a.K * 4, per_xcd, &blocks);
    launch_main(a.gate ? proj_gemm_lds_kernel<GROUPS, WN, RING, PIPE, KS, true> : proj_gemm_lds_kernel<GROUPS, WN, RING, PIPE, KS>,
                dim3(blocks), dim3(128 * WN * KS), a, gemm_lds_bytes<GROUPS, WN, RING, KS>());
}

// Register tiles: the one whose estimate is the least.  A tile of NT x GROUPS waits for NT + GROUPS KiB a k-step
// through a compute unit's vector cache, workgroup after workgroup; an LDS tile of two sets of waves for as long as 17
// of them (from 1024 inputs on).  Chosen by workgroups alone before, wide weights took tiles too small (64 rows, 4096 ->
// 8192: 52 us in tiles of 32 x 16, 30 in 64 x 32; 160 rows 65, 41; 1500 rows, 5120 -> 1024 86, 66).  Over 15 row counts
// from 17 to 1500, 10 input ranges and 7 widths (profiles/projection_product_forms.txt has every form's time) the form
// picked is 1.4 % off the best one on average, 24 % (1.3 us of 5.4) at worst.
// The gated tiles follow the plain ones in the choice between registers and LDS: only then do both take the same sums
// (a register tile of any size has the same ones), and the gated product the bits of the plain one's activation.
void launch_proj_tiles(const ProjArgs& a, uint32_t groups)
{
    struct Form {
        uint32_t groups, nt;
        void (*launch)(const ProjArgs&, uint32_t);
    };
    static const Form plain[] = {{1, 1, launch_proj_gemm_split<1, 1, 8>}, {2, 1, launch_proj_gemm_split<2, 1, 8>},
                                 {2, 2, launch_proj_gemm_split<2, 2, 8>}, {4, 2, launch_proj_gemm_split<4, 2, 4>},
                                 {4, 4, launch_proj_gemm_split<4, 4, 2>}},
                      gated[] = {{1, 2, launch_proj_gemm_split<1, 2, 8, true>}, {2, 2, launch_proj_gemm_split<2, 2, 8, true>},
                                 {4, 2, launch_proj_gemm_split<4, 2, 4, true>}, {4, 4, launch_proj_gemm_split<4, 4, 2, true>}};
    const uint32_t nt = a.N / 16;
    const auto rounds = [&](uint32_t w, uint32_t h) {
        return (uint32_t)(((uint64_t)((nt + w - 1) / w) * ((groups + h - 1) / h) + g.n_cus - 1) / g.n_cus);
    };
    uint32_t least = ~0u;
    const Form* best = nullptr;
    const auto offer = [&](const Form& f) {
        const uint32_t cost = rounds(f.nt, f.groups) * (f.nt + f.groups);
        if (cost < least) {
            least = cost;
            best = &f;
        }
    };
    for (const Form& f : plain) offer(f);
    if (a.K >= 1024 && a.K % 64 == 0 && rounds(8, 8) * 17 < least) {
        launch_proj_lds<4, 2, 4, true, 2>(a, groups, 32);
        return;
    }
    if (a.gate) {
        least = ~0u;
        for (const Form& f : gated) offer(f);
    }
    best->launch(a, groups);
}

void launch_proj_gemm(const ProjArgs& a, uint32_t groups)
{
    const uint32_t nt = a.N / 16, panels = (nt + 7) / 8;
    const uint32_t wide = (nt + 15) / 16;
    // The eight-wave tile runs one workgroup per CU, in rounds of 256: when its
    // last round would leave more than 10 % of the CUs idle, the four-wave tile
    // (two per CU, half the work each) loses less (2047 rows x 6144 outputs:
    // 384 eight-wave tiles, 1.5 rounds, 83 us; 768 four-wave tiles 65 us.
    // 1024 rows x 28672 outputs: 896 eight-wave tiles, 3.5 rounds, 559 us;
    // 1792 four-wave tiles 530 us).
    const uint32_t n_wide = wide * ((groups + 15) / 16), n_big = panels * ((groups + 15) / 16);
    const uint32_t rounds = (n_wide + 255) / 256;
    const bool wide_fills = n_wide >= 256 && (n_wide * 100 >= rounds * 256 * 90 || n_big < 512);
    // The four-wave tiles run two per CU, in rounds of 512.  The 128 x 128 tile moves
    // fewer bytes per MFMA than the 128 x 64 one (2048 rows x 4096 -> 6144: 226 against
    // 243 us) but has half as many workgroups to fill its last round with: where that
    // round would be thin (under 70 % full) and the smaller tile's is fuller by a tenth
    // or more, the smaller tile wins (1536 rows x 1024 -> 6144: 576 tiles, 1.1 rounds,
    // 59.8 us; 1152 smaller ones 49 us.  At three quarters full the larger tile still
    // holds its own: 2047 rows x 1024 -> 6144 65.6 against 64.8 us, 2048 x 4096 -> 6144
    // 226 against 243).
    const uint32_t n_small = panels * ((groups + 7) / 8);
    const uint32_t rounds_b = (n_big + 511) / 512, rounds_s = (n_small + 511) / 512;
    const bool small_fills_better = n_small >= 512 && n_big * 100 < rounds_b * 512 * 70 &&
                                    (uint64_t)n_small * rounds_b * 100 >= (uint64_t)n_big * rounds_s * 100 + (uint64_t)rounds_b * rounds_s * 512 * 10;
    if (wide_fills)
        launch_proj_lds<8, 4, 5, true, 1>(a, groups, 32);
    else if (n_big >= 512 && !small_fills_better)
        launch_proj_lds<8, 2, 3, false, 1>(a, groups, 64);
    else if (panels * ((groups + 7) / 8) >= 512)          // two and more per CU cover each other's latency
        launch_proj_lds<4, 2, 3, false, 1>(a, groups, 64);
    else if (panels * ((groups + 7) / 8) >= 256 && (a.K / 32) % 2 == 0 && a.K >= 2048)
        // one per CU and a long input range: two sets of waves halve it (two waves per SIMD, half the
        // chain of k-steps; 2047 rows x 2048 -> 1024: 40.3 -> 28.3 us, x 3072 -> 1024: 40 -> 36.6; at
        // 1024 inputs the sum through LDS costs more than the shorter chain gives)
        launch_proj_lds<4, 2, 4, true, 2>(a, groups, 32);
    else if (panels * ((groups + 7) / 8) >= 256)          // one per CU, one wave per SIMD: pipelined reads
        launch_proj_lds<4, 2, 4, true, 1>(a, groups, 32);
    else
        launch_proj_tiles(a, groups);
}

// proj_rows_fused_kernel<SRC, n_in / 128, nt>, or nullptr where none is built.
using FusedKernel = void (*)(const ProjArgs, const ProjPrepArgs);

template <int SRC, int D, int ROWS>
FusedKernel fused_of(uint32_t nt, bool gated)
{
    if (gated) {
        if constexpr (D <= 16)
            if (nt == 2) return proj_rows_fused_kernel<SRC, D, 2, true, ROWS>;
        if constexpr (D <= 8)
            if (nt == 4) return proj_rows_fused_kernel<SRC, D, 4, true, ROWS>;
        return nullptr;
    }
    if (nt == 1) return proj_rows_fused_kernel<SRC, D, 1, false, ROWS>;
    if constexpr (D <= 16)
        if (nt == 2) return proj_rows_fused_kernel<SRC, D, 2, false, ROWS>;
    if constexpr (D <= 8) {
        if (nt == 3) return proj_rows_fused_kernel<SRC, D, 3, false, ROWS>;
        if (nt == 4) return proj_rows_fused_kernel<SRC, D, 4, false, ROWS>;
    }
    return nullptr;
}

template <int ROWS>
FusedKernel fused_kernel(int src, uint32_t n_in, uint32_t nt, bool gated)
{
    const bool norm = src == kProjSrcRmsNorm;
    if (!norm && src != kProjSrcPlain) return nullptr;
    switch (n_in) {
    case 512: return norm ? fused_of<kProjSrcRmsNorm, 4, ROWS>(nt, gated) : fused_of<kProjSrcPlain, 4, ROWS>(nt, gated);
    case 1024: return norm ? fused_of<kProjSrcRmsNorm, 8, ROWS>(nt, gated) : fused_of<kProjSrcPlain, 8, ROWS>(nt, gated);
    case 1536: return norm ? fused_of<kProjSrcRmsNorm, 12, ROWS>(nt, gated) : fused_of<kProjSrcPlain, 12, ROWS>(nt, gated);
    case 2048: return norm ? fused_of<kProjSrcRmsNorm, 16, ROWS>(nt, gated) : fused_of<kProjSrcPlain, 16, ROWS>(nt, gated);
    case 2560: return norm ? nullptr : fused_of<kProjSrcPlain, 20, ROWS>(nt, gated);
    case 3072: return norm ? nullptr : fused_of<kProjSrcPlain, 24, ROWS>(nt, gated);
    default: return nullptr;
    }
}

// The kernel that makes its own operand fragments, and its tiles per workgroup: the
// fewest with which the launch is one workgroup per CU at most.  A second workgroup on
// a CU would make the same rows' terms again, and that is vector-ALU time nothing
// hides: 16 rows, norm + 1024 -> 4096, one / two / three / four tiles (512 / 256 / 172 /
// 128 workgroups) 6.7 / 5.2 / 5.9 / 6.5 us; -> 6144 8.6 / 7.8 / 6.2 / 6.8.
//
// Rows: four to a workgroup where there are CUs for it, eight otherwise, at the same number of tiles.  Halving the rows
// for twice the tiles would double the weights that a CU has to take in (46 bytes a nanosecond at best): not done.
//
// Gated weights of 17 to 40 rows that are too wide for that have a second workgroup on a CU, of four tiles and eight rows each, which is built
// for 512 and 1024 inputs: the launch that makes the fragments costs more than terms made twice (norm, us, apart / so: 1024 -> 2 x
// 2048, 33 rows 8.9 / 7.7; -> 2 x 3072, 17 rows 9.6 / 8.3, 32 9.8 / 8.8, 40 11.3 / 8.9; -> 2 x 5120, 24 rows 12.6 / 10.0; 512 -> 2 x
// 3072, 40 rows 8.8 / 5.6; without a norm 1024 -> 2 x 4096, 24 rows 8.5 / 8.8, 32 8.7 / 8.8, the others gain 2 to 33 %).
// Where one workgroup of four tiles fits, two of two tiles lose (1024 -> 2 x 1536, 24 rows 6.1 / 6.9; 2048 -> 2 x 2048 11.3 /
// 14.9), and so do weights that are not gated (1024 -> 4096, 32 rows 6.6 / 7.7, 3072 -> 1024, 40 rows 9.6 / 13.5).
FusedKernel pick_fused(int src, uint32_t n_in, uint32_t tiles, uint32_t rows, bool gated, uint32_t* nt, uint32_t* wg_rows)
{
    for (*nt = gated ? 2 : 1; *nt <= 4; *nt += gated ? 2 : 1)
        for (*wg_rows = 4; *wg_rows <= 8; *wg_rows *= 2)
            if ((tiles + *nt - 1) / *nt * ((rows + *wg_rows - 1) / *wg_rows) <= (uint32_t)g.n_cus)
                return *wg_rows == 4 ? fused_kernel<4>(src, n_in, *nt, gated) : fused_kernel<8>(src, n_in, *nt, gated);
    *nt = 4;
    *wg_rows = 8;
    if (gated && rows > 16 && rows <= 40 && (tiles + 3) / 4 * ((rows + 7) / 8) <= 2 * (uint32_t)g.n_cus) return fused_kernel<8>(src, n_in, 4, true);
    return nullptr;
}

// What feeds a projection: the rows as they are, their RMS normalisation, or
// the gated activation of rows that hold gate and up values side by side.
struct ProjSource {
    int kind = kProjSrcPlain;
    const float* norm_w = nullptr;
    float eps = 0.f;
    int gate = 0;            // kProjSrcSwiglu, kProjSrcGeglu: the weight's halves are gates and values (GATED kernels)
};

// Waves that share a run of outputs (contiguous parts of the inputs, summed
// through LDS in a fixed order): enough that a narrow weight still gives
// one to two thousand waves.  A function of the weight's shape only: a row's
// sums are then split the same way whether it travels alone or with up to
// fifteen others, so a batched step's rows equal the serial steps' bit
// for bit (reference contract: src/core/batch.c:15-19).  From 17 rows on the
// kernels have splits of their own.
uint32_t proj_ksplit(const wr_hip_weight* w)
{
    const uint32_t tiles = w->n_out / 16, ktiles = w->n_in / 32;
    uint32_t ksplit = 1;
    while (ksplit < 4 && tiles * ksplit < 2048 && ktiles % (ksplit * 2) == 0 &&
           ktiles / (ksplit * 2) >= 4)
        ksplit *= 2;
    return ksplit;
}

// y_dev[rows][ldy] = source(x_dev)[rows][n_in] . W^T (+ add_dev), rows <= kProjMaxRows;
// or, with `down`, into those rows of host memory (2 to 16, a weight of ksplit 1).  The caller has entered.
int proj_chunk_locked(const wr_hip_weight* w, uint32_t rows, const float* x_dev, uint32_t ldx,
                      const ProjSource& src, const float* add_dev, float* y_dev, uint32_t ldy,
                      const ProjDownArgs* down = nullptr)
{
    cx->rows.store(rows, std::memory_order_relaxed);
    const uint32_t groups = (rows + 7) / 8;                // row groups of eight
    const bool gemm = rows >= (uint32_t)kProjGemmMinRows;
    const uint32_t ktiles = w->n_in / 32;
    // The kernels that make the operand terms themselves read the rows while others already write results.
    const uint32_t x_cols = src.kind == kProjSrcSwiglu || src.kind == kProjSrcGeglu ? 2 * w->n_in : w->n_in;
    const uint32_t y_cols = src.gate ? w->n_out / 2 : w->n_out;
    const uintptr_t x0 = (uintptr_t)x_dev, y0 = (uintptr_t)y_dev;
    const bool apart = x0 + ((size_t)(rows - 1) * ldx + x_cols) * 4 <= y0 || y0 + ((size_t)(rows - 1) * ldy + y_cols) * 4 <= x0;
    // one row: the fragment step runs inside the product's kernel (4 bytes of LDS per input)
    const bool row1 = !down && rows == 1 && apart && (size_t)w->n_in * 4 <= kProjRow1MaxLds;
    const uint32_t tiles = w->n_out / 16, ksplit = groups <= 2 ? proj_ksplit(w) : 1;
    // up to a few dozen rows, where one workgroup per CU can take them all: so does each workgroup of the product.  It
    // reads the rows with 16-byte loads.
    // (Four waves to the inputs, as the kernel of one row then has: a row's bits are its own in a step of up to sixteen.)
    uint32_t fused_nt = 0, fused_rows = 0;
    const FusedKernel fused =
        !down && rows > 1 && rows < kProjGroupRows && (gemm || ksplit == 4) && ldx % 4 == 0 && ((x0 | (uintptr_t)src.norm_w) & 15) == 0 && apart
            ? pick_fused(src.kind, w->n_in, tiles, rows, src.gate != 0, &fused_nt, &fused_rows)
            : nullptr;
    const size_t frag_bytes = (size_t)groups * ktiles * 1024;
    int rc = ensure_device(cx->d_proj, frag_bytes + kProjMaxRows * sizeof(float));
    if (rc) return rc;
    half8* frag = reinterpret_cast<half8*>(cx->d_proj.p);
    float* scales = reinterpret_cast<float*>((uint8_t*)cx->d_proj.p + frag_bytes);
    ProjPrepArgs pa;
    pa.x = x_dev;
    pa.norm_w = src.norm_w;
    pa.frag = frag;
    pa.scales = scales;
    pa.ldx = ldx;
    pa.R = rows;
    pa.K = w->n_in;
    pa.eps = src.eps;
    const dim3 pgrid(groups * 8), pblock(256);
    const bool in_regs = w->n_in <= 4096;           // two chunks of eight values per thread
    // many rows: a workgroup per row group (whole-line writes); it reads rows
    // with 16-byte loads
    const bool by_group = rows >= kProjGroupRows && ldx % 4 == 0 && ((uintptr_t)x_dev & 15) == 0 &&
                          ((uintptr_t)src.norm_w & 15) == 0;
    const uint32_t kin = w->n_in;
#define WR_LAUNCH_PREP_GROUP(SRC, CH) \
    hipLaunchKernelGGL(HIP_KERNEL_NAME(proj_prep_group_kernel<SRC, CH>), dim3(groups), pblock, 0, cx->stream, pa)
#define WR_LAUNCH_PREP(SRC)                                                                          \
    do {                                                                                             \
        if (by_group && kin <= 1024)                                                                 \
            WR_LAUNCH_PREP_GROUP(SRC, 4);                                                            \
        else if (by_group && kin <= 2048)                                                            \
            WR_LAUNCH_PREP_GROUP(SRC, 8);                                                            \
        else if (by_group && kin <= 4096)                                                            \
            WR_LAUNCH_PREP_GROUP(SRC, 16);                                                           \
        else if (by_group)                                                                           \
            WR_LAUNCH_PREP_GROUP(SRC, 0);                                                            \
        else if (in_regs)                                                                            \
            hipLaunchKernelGGL(HIP_KERNEL_NAME(proj_prep_kernel<SRC, 2>), pgrid, pblock, 0, cx->stream, pa); \
        else                                                                                         \
            hipLaunchKernelGGL(HIP_KERNEL_NAME(proj_prep_kernel<SRC, 0>), pgrid, pblock, 0, cx->stream, pa); \
    } while (0)
    if (row1 || fused)
        ;                                           // no fragment launch
    else if (src.kind == kProjSrcRmsNorm)
        WR_LAUNCH_PREP(kProjSrcRmsNorm);
    else if (src.kind == kProjSrcSwiglu)
        WR_LAUNCH_PREP(kProjSrcSwiglu);
    else if (src.kind == kProjSrcGeglu)
        WR_LAUNCH_PREP(kProjSrcGeglu);
    else
        WR_LAUNCH_PREP(kProjSrcPlain);
#undef WR_LAUNCH_PREP
#undef WR_LAUNCH_PREP_GROUP
    ProjArgs a;
    a.w = reinterpret_cast<const half8*>(w->tiles);
    a.xfrag = frag;
    a.scales = scales;
    a.bias_rows = add_dev;
    a.y = y_dev;
    a.N = w->n_out;
    a.K = w->n_in;
    a.R = rows;
    a.ldy = ldy;
    a.gate = (uint8_t)src.gate;
    a.ksplit = (uint8_t)ksplit;
    if (down) {
        const dim3 grid((tiles + 7) / 8);
        launch_main(groups == 1 ? proj_rows_down_kernel<1> : proj_rows_down_kernel<2>, grid, dim3(kProjThreads), a, *down, kOnePerCuLds);
    } else if (row1) {
        const uint32_t per_block = 4 / ksplit, pair_blocks = (tiles / 2 + per_block - 1) / per_block;
        const bool pairs = src.gate && pair_blocks * 2 > g.n_cus;
        const dim3 grid(pairs ? pair_blocks : (tiles + per_block - 1) / per_block), block(kProjThreads);
        const size_t lds = (size_t)w->n_in * 4;
        if (pairs && src.kind == kProjSrcRmsNorm)
            launch_main(proj_row1_kernel<kProjSrcRmsNorm, kRow1Gated>, grid, block, a, pa, lds);
        else if (pairs)
            launch_main(proj_row1_kernel<kProjSrcPlain, kRow1Gated>, grid, block, a, pa, lds);
        else if (src.gate && src.kind == kProjSrcRmsNorm)
            launch_main(proj_row1_kernel<kProjSrcRmsNorm, kRow1GatedHalf>, grid, block, a, pa, lds);
        else if (src.gate)
            launch_main(proj_row1_kernel<kProjSrcPlain, kRow1GatedHalf>, grid, block, a, pa, lds);
        else if (src.kind == kProjSrcRmsNorm)
            launch_main(proj_row1_kernel<kProjSrcRmsNorm>, grid, block, a, pa, lds);
        else if (src.kind == kProjSrcSwiglu)
            launch_main(proj_row1_kernel<kProjSrcSwiglu>, grid, block, a, pa, lds);
        else if (src.kind == kProjSrcGeglu)
            launch_main(proj_row1_kernel<kProjSrcGeglu>, grid, block, a, pa, lds);
        else
            launch_main(proj_row1_kernel<kProjSrcPlain>, grid, block, a, pa, lds);
    } else if (fused)
        launch_main(fused, dim3((tiles + fused_nt - 1) / fused_nt, (rows + fused_rows - 1) / fused_rows), dim3(kProjThreads), a, pa, (size_t)w->n_in * 32);
    else if (gemm)
        launch_proj_gemm(a, groups);
    else if (src.gate && groups == 1)
        launch_proj<1, 2, true>(a);
    else if (src.gate)
        launch_proj<2, 2, true>(a);
    else if (ksplit == 4 && !(w->n_in > 4096 && (uint64_t)w->n_in * w->n_out >= 12u << 20)) {
        // A workgroup per tile and group of eight rows, four waves to the input range: the
        // same parts in the same order as below, so the same bits.  For 9 .. 16 rows the
        // weights pass L2 twice, but a workgroup reads half the operand fragments, which
        // at 16 rows are twice the weights' bytes: 16 rows, weights from HBM, 1024 -> 4096
        // 4.7 -> 4.2 us, 2048 -> 1024 5.3 -> 4.3, 1024 -> 6144 6.0 -> 5.4, 3072 -> 1024
        // 7.0 -> 5.5 (4 rows: 4.2 -> 3.7, 4.4, 5.2 -> 4.9, 5.9 -> 5.6).  Where the tiles are
        // more than the CUs the weights' second pass is the larger loss: 32 x 16 (16 rows,
        // 4096 -> 8192 26.6 us in tiles of 16 x 8, 22.4 below, 22.1; 2048 -> 6144 12.4, 12.6,
        // 11.3).  Long ranges of large weights stream faster below: 8192 -> 4096 34.4 us
        // against 25.9, 14 336 -> 8192 101 against 55 (4 rows 27.0, 22.0; 61, 52); the line
        // lies between 5120 -> 2048 (13.7 us, 14.3 below) and 6144 -> 2048 (18.4, 15.8).
        if (groups == 2 && tiles > g.n_cus)
            launch_proj_gemm_split<2, 2, 8>(a, groups);
        else
            launch_proj_gemm_split<1, 1, 8>(a, groups);
    } else if (groups == 1)
        launch_proj<1, 1>(a);
    else if (tiles * ksplit >= 2048)
        launch_proj<2, 2>(a);               // wide weight: two output tiles per operand load
    else
        launch_proj<2, 1>(a);               // narrow weight: every wave counts
    HIP_TRY(hipGetLastError(), "projection launch", 0);
    return WR_HIP_OK;
}

int proj_locked(const wr_hip_weight* w, uint32_t rows, const float* x_dev, uint32_t ldx,
                const ProjSource& src, const float* add_dev, float* y_dev, uint32_t ldy)
{
    for (uint32_t done = 0; done < rows; done += kProjMaxRows) {
        const uint32_t n = rows - done < (uint32_t)kProjMaxRows ? rows - done : (uint32_t)kProjMaxRows;
        int rc = proj_chunk_locked(w, n, x_dev + (size_t)done * ldx, ldx, src,
                                   add_dev ? add_dev + (size_t)done * ldy : nullptr,
                                   y_dev + (size_t)done * ldy, ldy);
        if (rc) return rc;
    }
    return WR_HIP_OK;
}

}  // namespace

// ======================================================================= ABI

extern "C" {

int wr_hip_attn_init(int device)
{
    std::lock_guard<std::mutex> lk(g.mu);
    if (g.inited) return WR_HIP_ERR_STATE;
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count <= 0) {
        logmsg(0, "init: no HIP device visible; this library has no CPU path");
        return WR_HIP_ERR_UNSUPPORTED;
    }
    if (device < 0 || device >= count) return WR_HIP_ERR_INVAL;
    hipDeviceProp_t prop;
    HIP_TRY(hipSetDevice(device), "set device", 0);
    HIP_TRY(hipGetDeviceProperties(&prop, device), "device properties", 0);
    if (strncmp(prop.gcnArchName, "gfx950", 6) != 0) {
        logmsg(0, "init: device %d is %s; the kernels are built for gfx950 only", device,
               prop.gcnArchName);
        return WR_HIP_ERR_UNSUPPORTED;
    }
    g.device = device;
    g.n_cus = prop.multiProcessorCount > 0 ? (uint32_t)prop.multiProcessorCount : 256u;
    snprintf(g.name, sizeof g.name, "%s %s, %d CUs, %.1f GiB", prop.gcnArchName, prop.name,
             prop.multiProcessorCount, (double)prop.totalGlobalMem / (1024.0 * 1024.0 * 1024.0));
    g.inited = true;
    g.calls.store(0);
    {
        const char* e = getenv("WR_HIP_PREFILL_TWO_WAVES");
        g.prefill_two_waves = (e && e[0] == '0') ? 0 : 1;
        e = getenv("WR_HIP_PREFILL_PART_MB");
        g.prefill_part_mb = e && e[0] ? (uint32_t)std::min(strtoul(e, nullptr, 10), (unsigned long)kMaxPrefillPartMb) : kMaxPrefillPartMb;
        e = getenv("WR_HIP_PREFILL_256_FOUR_WAVES");
        g.prefill_256_four_waves = (e && e[0] == '1') ? 1 : 0;
    }
    g.generation++;
    int rc = WR_HIP_OK;
    {
        const hipError_t e = hipEventCreateWithFlags(&g.noalloc_done, hipEventDisableTiming);
        if (e != hipSuccess) rc = hip_fail(e, "event create", 0);
        g.noalloc_recorded = false;
    }
    if (rc == WR_HIP_OK) {
        // device address of the no-alloc entry point's scratch array, once per
        // device, with that device current
        if (device >= kMaxDevices) {
            rc = WR_HIP_ERR_LIMIT;
        } else if (!g.noalloc_ws[device]) {
            void* p = nullptr;
            hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
            if (e != hipSuccess || !p)
                rc = hip_fail(e, "address of the no-alloc scratch array", 0);
            else
                g.noalloc_ws[device] = reinterpret_cast<unsigned char*>(p);
        }
    }
    if (rc == WR_HIP_OK) {
        hipError_t e = hipSuccess;
        const auto allow_lds = [&](auto kernel, size_t bytes) {
            if (kernel && e == hipSuccess)
                e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        };
        // the prefill kernels stage more than the 64 KiB a kernel may use without asking
        allow_lds(prefill_il_kernel<64, 4, false>, split_smem_bytes<64, 4>());
        allow_lds(prefill_il_kernel<64, 4, true>, split_smem_bytes<64, 4>());
        allow_lds(prefill_il_kernel<64, 2, false>, split_smem_bytes<64, 2>());
        allow_lds(prefill_il_kernel<64, 2, true>, split_smem_bytes<64, 2>());
        allow_lds(prefill_il_kernel<128, 4, false>, split_smem_bytes<128, 4>());
        allow_lds(prefill_il_kernel<128, 4, true>, split_smem_bytes<128, 4>());
        allow_lds(prefill_il_kernel<128, 2, false>, split_smem_bytes<128, 2>());
        allow_lds(prefill_il_kernel<128, 2, true>, split_smem_bytes<128, 2>());
        allow_lds(prefill_ild_kernel<4, false>, ild_smem_bytes<4>());
        allow_lds(prefill_ild_kernel<4, true>, ild_smem_bytes<4>());
        allow_lds(prefill_ild_kernel<2, false>, ild_smem_bytes<2>());
        allow_lds(prefill_ild_kernel<2, true>, ild_smem_bytes<2>());
        allow_lds(prefill_pair_kernel<128, false>, pair_smem_bytes<128>());
        allow_lds(prefill_pair_kernel<128, true>, pair_smem_bytes<128>());
        // (a gated row: 6 KiB of partial tiles beside its terms, more than 64 KiB together from 14 848 inputs on)
        allow_lds(proj_rows_down_kernel<1>, kOnePerCuLds);
        allow_lds(proj_rows_down_kernel<2>, kOnePerCuLds);
        allow_lds(proj_row1_kernel<kProjSrcRmsNorm, kRow1Gated>, kProjRow1MaxLds);
        allow_lds(proj_row1_kernel<kProjSrcPlain, kRow1Gated>, kProjRow1MaxLds);
        allow_lds(proj_gemm_lds_kernel<8, 4, 5, true>, gemm_lds_bytes<8, 4, 5>());
        allow_lds(proj_gemm_lds_kernel<8, 4, 5, true, 1, true>, gemm_lds_bytes<8, 4, 5>());
        allow_lds(proj_gemm_lds_kernel<8, 2, 3>, gemm_lds_bytes<8, 2, 3>());
        allow_lds(proj_gemm_lds_kernel<8, 2, 3, false, 1, true>, gemm_lds_bytes<8, 2, 3>());
        allow_lds(proj_gemm_lds_kernel<4, 2, 4, true>, gemm_lds_bytes<4, 2, 4>());
        allow_lds(proj_gemm_lds_kernel<4, 2, 4, true, 1, true>, gemm_lds_bytes<4, 2, 4>());
        allow_lds(proj_gemm_lds_kernel<4, 2, 4, true, 2>, gemm_lds_bytes<4, 2, 4, 2>());
        allow_lds(proj_gemm_lds_kernel<4, 2, 4, true, 2, true>, gemm_lds_bytes<4, 2, 4, 2>());
        for (uint32_t n_in = 512; n_in <= 3072; n_in += 512)
            for (uint32_t nt = 1; nt <= 4; nt++)
                for (const int src : {kProjSrcPlain, kProjSrcRmsNorm})
                    for (const bool gated : {false, true}) {
                        allow_lds(fused_kernel<4>(src, n_in, nt, gated), (size_t)n_in * 32);
                        allow_lds(fused_kernel<8>(src, n_in, nt, gated), (size_t)n_in * 32);
                    }
        if (e != hipSuccess) rc = hip_fail(e, "kernel LDS size", 0);
    }
    if (rc != WR_HIP_OK) {
        g.inited = false;
        if (g.noalloc_done) (void)hipEventDestroy(g.noalloc_done);
        g.noalloc_done = nullptr;
    }
    return rc;
}

void wr_hip_attn_shutdown(void)
{
    std::lock_guard<std::mutex> lk(g.mu);
    if (!g.inited) return;
    (void)hipSetDevice(g.device);
    for (Ctx* c : g.ctxs) ctx_destroy(c);      // waits for each stream first
    g.ctxs.clear();
    g.idle.clear();
    cx = nullptr;
    {
        std::lock_guard<std::mutex> kept(g.slab_mu);
        for (const Lib::Slab& s : g.slabs) (void)hipFree(s.p);
        g.slabs.clear();
    }
    if (g.noalloc_done) (void)hipEventDestroy(g.noalloc_done);
    g.noalloc_done = nullptr;
    g.inited = false;
    g.device = -1;
    g.tune_keys_per_wg = 0;
    g.force_generic = 0;
    g.step_owner = nullptr;
    g.step_refused = 0;
    g.step_limit = 0;
    g.fail_allocs = 0;
}

void wr_hip_attn_set_log(wr_hip_log_fn fn, void* user)
{
    g.log_fn = fn;
    g.log_user = user;
}

uint64_t wr_hip_attn_calls(void) { return g.calls.load(std::memory_order_relaxed); }

const char* wr_hip_attn_device_name(void) { return g.name; }

uint32_t wr_hip_attn_caps(void) { return WR_HIP_CAP_PROJ; }

void wr_hip_attn_set_prefill_part_mb(uint32_t mb) { g.prefill_part_mb = std::min(mb, kMaxPrefillPartMb); }

void wr_hip_attn_set_prefill_one_wave(int on)
{
    g.prefill_two_waves = on ? 0 : 1;
}

void wr_hip_attn_set_tuning(uint32_t decode_keys_per_wg, int force_generic)
{
    std::lock_guard<std::mutex> lk(g.mu);
    g.tune_keys_per_wg = decode_keys_per_wg;
    g.force_generic = force_generic;
}

// ---------------------------------------------------------------- storage --

int wr_hip_attn_kv_create(uint32_t n_layers, const uint32_t* hd_per_layer, uint32_t nkv,
                          uint32_t max_ctx, wr_hip_kv** out)
{
    if (!out) return WR_HIP_ERR_INVAL;
    *out = nullptr;
    if (!g.inited) return WR_HIP_ERR_STATE;
    if (!hd_per_layer || n_layers == 0 || nkv == 0 || max_ctx == 0) return WR_HIP_ERR_INVAL;
    if (n_layers > WR_HIP_MAX_LAYERS) return WR_HIP_ERR_LIMIT;
    if (max_ctx > WR_HIP_ATTN_MAX_SEQ) return WR_HIP_ERR_LIMIT;
    for (uint32_t L = 0; L < n_layers; L++)
        if (hd_per_layer[L] > WR_HIP_FLASH_D_MAX) return WR_HIP_ERR_LIMIT;

    wr_hip_kv* kv = new (std::nothrow) wr_hip_kv();
    if (!kv) return WR_HIP_ERR_NOMEM;
    kv->n_layers = n_layers;
    kv->nkv = nkv;
    kv->max_ctx = max_ctx;
    kv->ctx_pad = (max_ctx + kVBlock - 1) / kVBlock * kVBlock;
    size_t cur = 0;
    bool any = false;
    for (uint32_t L = 0; L < n_layers; L++) {
        kv->hd[L] = hd_per_layer[L];
        if (kv->hd[L] == 0) continue;
        any = true;
        // K rows are padded to whole 16-byte chunks (common.hip.h); Vt is not
        const size_t k_side = ((size_t)nkv * kv->ctx_pad * k_padded_hd(kv->hd[L]) * 2 + 255) & ~(size_t)255;
        const size_t v_side = ((size_t)nkv * kv->ctx_pad * kv->hd[L] * 2 + 255) & ~(size_t)255;
        kv->k_off[L] = cur;
        cur += k_side;
        kv->vt_off[L] = cur;
        cur += v_side;
    }
    if (!any) {
        delete kv;
        return WR_HIP_ERR_INVAL;
    }
    kv->bytes = cur;

    ENTER();
    kv->device = g.device;
    Lib::Slab kept{};
    const bool again = slab_take(cur, kept);
    kv->slab = kept.p;
    hipError_t e = again ? hipSuccess : device_malloc((void**)&kv->slab, cur);
    if (e != hipSuccess) {
        logmsg(0, "session: device slab alloc failed (%zu bytes): %s", cur, hipGetErrorString(e));
        delete kv;
        return WR_HIP_ERR_NOMEM;
    }
    e = again ? slab_clear(kept) : hipMemsetAsync(kv->slab, 0, cur, cx->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(cx->stream);
    if (e != hipSuccess) {
        (void)hipFree(kv->slab);
        delete kv;
        return hip_fail(e, "slab clear", 0);
    }
    *out = kv;
    return WR_HIP_OK;
}

void wr_hip_attn_kv_destroy(wr_hip_kv* kv)
{
    if (!kv) return;
    if (g.inited) {
        Entered entered_;
        if (entered_.ok()) (void)hipStreamSynchronize(cx->stream);
        if (kv->slab && entered_.ok() && kv->device == g.device) slab_leave(kv);
        else if (kv->slab) (void)hipFree(kv->slab);          // (waits for the device's other streams by itself)
    }
    delete kv;
}

void wr_hip_attn_trim(void)
{
    if (!g.inited) return;
    Entered entered_;
    if (entered_.ok()) (void)slabs_trim();
}

uint64_t wr_hip_attn_kv_bytes(const wr_hip_kv* kv) { return kv ? kv->bytes : 0; }

// ----------------------------------------------------------------- append --

int wr_hip_attn_append_dev(wr_hip_kv* kv, uint32_t layer, uint32_t pos, uint32_t n_rows,
                           const float* k_f32_dev, const float* v_f32_dev)
{
    int rc = check_append(kv, layer, pos, n_rows, k_f32_dev, v_f32_dev);
    if (rc || n_rows == 0) return rc;
    ENTER();
    return append_rows_locked<float>(kv, layer, pos, n_rows, k_f32_dev, v_f32_dev);
}

int wr_hip_attn_append_batched_dev(uint32_t n, wr_hip_kv* const* kv, uint32_t layer,
                                   const uint32_t* pos, const float* k_f32_dev,
                                   const float* v_f32_dev)
{
    if (!g.inited) return WR_HIP_ERR_STATE;
    if (!kv || !pos || !k_f32_dev || !v_f32_dev) return WR_HIP_ERR_INVAL;
    if (n == 0 || n > WR_HIP_BATCH_MAX) return WR_HIP_ERR_LIMIT;
    AppendBatchArgs a;
    memset(&a, 0, sizeof a);
    for (uint32_t i = 0; i < n; i++) {
        int rc = check_layer(kv[i], layer);
        if (rc) return rc;
        if (kv[i]->nkv != kv[0]->nkv || kv[i]->hd[layer] != kv[0]->hd[layer]) return WR_HIP_ERR_INVAL;
        for (uint32_t j = 0; j < i; j++)
            if (kv[i] == kv[j]) return WR_HIP_ERR_INVAL;
        if (pos[i] >= kv[i]->max_ctx) return WR_HIP_ERR_CTX_FULL;      // nothing is written
        a.k[i] = reinterpret_cast<uint16_t*>(kv[i]->slab + kv[i]->k_off[layer]);
        a.vt[i] = reinterpret_cast<uint16_t*>(kv[i]->slab + kv[i]->vt_off[layer]);
        a.pos[i] = pos[i];
        a.ctx_pad[i] = kv[i]->ctx_pad;
    }
    a.k_src = k_f32_dev;
    a.v_src = v_f32_dev;
    a.nkv = kv[0]->nkv;
    a.hd = kv[0]->hd[layer];
    ENTER();
    for (uint32_t i = 0; i < n; i++) kv[i]->writes((uint64_t)pos[i] + 1);
    hipLaunchKernelGGL(append_batch_kernel, dim3(n), dim3(256), 0, cx->stream, a);
    HIP_TRY(hipGetLastError(), "batched append launch", layer);
    return WR_HIP_OK;
}

int wr_hip_attn_rope_dev(void* x_dev, const void* cos_sin_dev, uint32_t rows, uint32_t heads,
                         uint32_t hd, uint32_t n_rot)
{
    if (!g.inited) return WR_HIP_ERR_STATE;
    if (!x_dev || !cos_sin_dev) return WR_HIP_ERR_INVAL;
    if (hd < 2 || (hd & 1) || heads == 0 || n_rot > hd / 2) return WR_HIP_ERR_INVAL;
    if (rows == 0 || n_rot == 0) return WR_HIP_OK;
    ENTER();
    const size_t total = (size_t)rows * heads * n_rot;
    hipLaunchKernelGGL(rope_rows_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                       cx->stream, reinterpret_cast<float*>(x_dev),
                       reinterpret_cast<const float*>(cos_sin_dev), rows, heads, hd, n_rot);
    HIP_TRY(hipGetLastError(), "rope launch", 0);
    return WR_HIP_OK;
}

int wr_hip_attn_rope_table_dev(float* cos_sin_dev, uint32_t rows, uint32_t pos0,
                               const uint32_t* pos, uint32_t hd, float theta_base,
                               uint32_t n_rot_pairs)
{
    if (!g.inited) return WR_HIP_ERR_STATE;
    if (!cos_sin_dev || rows == 0) return WR_HIP_ERR_INVAL;
    if (hd < 2 || (hd & 1)) return WR_HIP_ERR_INVAL;
    if (pos && rows > WR_HIP_BATCH_MAX) return WR_HIP_ERR_INVAL;
    // The kernel folds an angle into [-pi, pi] by subtracting 2 pi turn by turn, as
    // the reference does (src/core/mathx.c:112-147); from an angle of 2^27 on a
    // float's spacing exceeds 2 pi, the subtraction rounds back to itself and the
    // turns never end.  The reference's callers stay below WR_ATTN_MAX_SEQ: the
    // same bound here, before anything is launched.
    if (!pos && (uint64_t)pos0 + rows > WR_HIP_ATTN_MAX_SEQ) return WR_HIP_ERR_LIMIT;
    for (uint32_t i = 0; pos && i < rows; i++)
        if (pos[i] >= WR_HIP_ATTN_MAX_SEQ) return WR_HIP_ERR_LIMIT;
    RopeTableArgs a{};
    a.out = cos_sin_dev;
    a.rows = rows;
    a.hd = hd;
    a.n_rot = (n_rot_pairs >= 1 && n_rot_pairs < hd / 2) ? n_rot_pairs : hd / 2;
    a.theta = theta_base < 1.0f ? 10000.0f : theta_base;
    a.pos0 = pos0;
    a.listed = pos ? 1u : 0u;
    for (uint32_t i = 0; pos && i < rows; i++) a.pos[i] = pos[i];
    ENTER();
    hipLaunchKernelGGL(rope_table_kernel, dim3((rows + 63u) / 64u, a.n_rot), dim3(64), 0, cx->stream, a);
    HIP_TRY(hipGetLastError(), "rotary table launch", 0);
    return WR_HIP_OK;
}

int wr_hip_attn_append_rope(wr_hip_kv* kv, uint32_t layer, uint32_t pos, uint32_t n_rows,
                            const float* k_f32, const float* v_f32, const float* cos_sin,
                            uint32_t n_rot)
{
    int rc = check_append(kv, layer, pos, n_rows, k_f32, v_f32);
    if (rc) return rc;
    if (!cos_sin && n_rot > 0) return WR_HIP_ERR_INVAL;
    if (n_rot > kv->hd[layer] / 2) return WR_HIP_ERR_INVAL;
    if (n_rows == 0) return WR_HIP_OK;
    const uint32_t hd = kv->hd[layer], nkv = kv->nkv;
    const size_t bytes = (size_t)n_rows * nkv * hd * sizeof(float);
    const size_t tbytes = (size_t)n_rows * n_rot * 2 * sizeof(float);
    ENTER();
    rc = ensure_device(cx->d_stage, 2 * bytes + tbytes);
    if (rc) return rc;
    float* dk = reinterpret_cast<float*>(cx->d_stage.p);
    float* dv = reinterpret_cast<float*>((uint8_t*)cx->d_stage.p + bytes);
    float* dt = reinterpret_cast<float*>((uint8_t*)cx->d_stage.p + 2 * bytes);
    rc = copy_up(dk, k_f32, bytes, 0);
    if (rc == WR_HIP_OK) rc = copy_up(dv, v_f32, bytes, bytes);
    if (rc == WR_HIP_OK) rc = copy_up(dt, cos_sin, tbytes, 2 * bytes);
    if (rc == WR_HIP_OK && n_rot > 0) {
        const size_t total = (size_t)n_rows * nkv * n_rot;
        hipLaunchKernelGGL(rope_rows_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                           cx->stream, dk, dt, n_rows, nkv, hd, n_rot);
        HIP_TRY(hipGetLastError(), "rope launch", layer);
    }
    if (rc == WR_HIP_OK) rc = append_rows_locked<float>(kv, layer, pos, n_rows, dk, dv);
    // the staging buffers are reused by the next call: wait for the kernels
    if (rc == WR_HIP_OK) HIP_TRY(hipStreamSynchronize(cx->stream), "append sync", layer);
    return rc;
}

int wr_hip_attn_append(wr_hip_kv* kv, uint32_t layer, uint32_t pos, uint32_t n_rows,
                       const float* k_f32, const float* v_f32)
{
    int rc = check_append(kv, layer, pos, n_rows, k_f32, v_f32);
    if (rc || n_rows == 0) return rc;
    const size_t bytes = (size_t)n_rows * kv->nkv * kv->hd[layer] * sizeof(float);
    ENTER();
    rc = ensure_device(cx->d_stage, 2 * bytes);
    if (rc) return rc;
    float* dk = reinterpret_cast<float*>(cx->d_stage.p);
    float* dv = reinterpret_cast<float*>((uint8_t*)cx->d_stage.p + bytes);
    rc = copy_up(dk, k_f32, bytes, 0);
    if (rc == WR_HIP_OK) rc = copy_up(dv, v_f32, bytes, bytes);
    if (rc == WR_HIP_OK) rc = append_rows_locked<float>(kv, layer, pos, n_rows, dk, dv);
    // the staging buffers are reused by the next call: wait for the kernels
    if (rc == WR_HIP_OK) HIP_TRY(hipStreamSynchronize(cx->stream), "append sync", layer);
    return rc;
}

int wr_hip_attn_kv_write(wr_hip_kv* kv, uint32_t layer, uint32_t pos, uint32_t n_rows,
                         const uint16_t* k_f16, const uint16_t* v_f16)
{
    int rc = check_append(kv, layer, pos, n_rows, k_f16, v_f16);
    if (rc || n_rows == 0) return rc;
    const size_t bytes = (size_t)n_rows * kv->nkv * kv->hd[layer] * sizeof(uint16_t);
    ENTER();
    rc = ensure_device(cx->d_stage, 2 * bytes);
    if (rc) return rc;
    uint16_t* dk = reinterpret_cast<uint16_t*>(cx->d_stage.p);
    uint16_t* dv = reinterpret_cast<uint16_t*>((uint8_t*)cx->d_stage.p + bytes);
    rc = copy_up(dk, k_f16, bytes, 0);
    if (rc == WR_HIP_OK) rc = copy_up(dv, v_f16, bytes, bytes);
    if (rc == WR_HIP_OK) rc = append_rows_locked<uint16_t>(kv, layer, pos, n_rows, dk, dv);
    if (rc == WR_HIP_OK) HIP_TRY(hipStreamSynchronize(cx->stream), "kv_write sync", layer);
    return rc;
}

int wr_hip_attn_kv_read(wr_hip_kv* kv, uint32_t layer, uint32_t pos, uint32_t n_rows,
                        uint16_t* k_f16, uint16_t* v_f16)
{
    if (!g.inited) return WR_HIP_ERR_STATE;
    int rc = check_layer(kv, layer);
    if (rc) return rc;
    if (n_rows == 0) return WR_HIP_OK;
    if (!k_f16 || !v_f16) return WR_HIP_ERR_INVAL;
    if ((uint64_t)pos + n_rows > kv->max_ctx) return WR_HIP_ERR_INVAL;
    const uint32_t hd = kv->hd[layer], nkv = kv->nkv;
    const size_t total = (size_t)n_rows * nkv * hd;
    const size_t bytes = total * sizeof(uint16_t);
    ENTER();
    rc = ensure_device(cx->d_stage, 2 * bytes);
    if (rc) return rc;
    uint16_t* dk = reinterpret_cast<uint16_t*>(cx->d_stage.p);
    uint16_t* dv = reinterpret_cast<uint16_t*>((uint8_t*)cx->d_stage.p + bytes);
    hipLaunchKernelGGL(export_kv_kernel, dim3((uint32_t)((total + 255) / 256)), dim3(256), 0,
                       cx->stream,
                       reinterpret_cast<const uint16_t*>(kv->slab + kv->k_off[layer]),
                       reinterpret_cast<const uint16_t*>(kv->slab + kv->vt_off[layer]), dk, dv, pos,
                       n_rows, nkv, hd, kv->ctx_pad);
    HIP_TRY(hipGetLastError(), "export launch", layer);
    rc = copy_down_sync(k_f16, dk, bytes);
    if (rc == WR_HIP_OK) rc = copy_down_sync(v_f16, dv, bytes);
    return rc;
}

// ----------------------------------------------------------------- decode --

int wr_hip_attn_decode_batched_dev(uint32_t n, wr_hip_kv* const* kv, uint32_t layer,
                                   const uint32_t* seq_k, const float* q_dev, float* out_dev,
                                   uint32_t nq, float scale_override, uint32_t window)
{
    int rc = check_decode(n, kv, layer, seq_k, q_dev, out_dev, nq);
    if (rc) return rc;
    ENTER();
    return decode_locked(n, kv, layer, seq_k, q_dev, out_dev, nq, scale_override, window);
}

int wr_hip_attn_decode_batched_dev_noalloc(uint32_t n, wr_hip_kv* const* kv, uint32_t layer,
                                           const uint32_t* seq_k, const float* q_dev,
                                           float* out_dev, uint32_t nq, float scale_override,
                                           uint32_t window)
{
    int rc = check_decode(n, kv, layer, seq_k, q_dev, out_dev, nq);
    if (rc) return rc;
    if (nq > kNoAllocMaxHeads) {
        logmsg(0, "decode (no-alloc form): %u query heads exceed the %u the fixed ticket array holds",
               nq, kNoAllocMaxHeads);
        return WR_HIP_ERR_LIMIT;
    }
    // A thread's first call into the library makes its stream and staging
    // buffers (hipStreamCreate, hipMalloc, hipHostMalloc): that call cannot be
    // this one.  Any other entry point (wr_hip_attn_sync is enough) does it.
    if (!t_slot.c || t_slot.generation != g.generation) {
        logmsg(0, "decode (no-alloc form): the calling thread has no stream context yet; "
                  "make one other library call from it first (wr_hip_attn_sync will do)");
        return WR_HIP_ERR_STATE;
    }
    ENTER();
    DecodeWorkspace fixed;
    fixed.ws = g.noalloc_ws[g.device];
    fixed.ticket_bytes = kNoAllocTicketBytes;
    fixed.bytes = kNoAllocScratchBytes;
    if (!fixed.ws) return WR_HIP_ERR_STATE;
    // One array per device, whatever thread calls: this launch waits for the
    // previous one that used it (on whichever stream that was), and leaves its
    // own mark for the next.  Event waits and records allocate nothing.
    std::lock_guard<std::mutex> chain(g.noalloc_mu);
    if (g.noalloc_recorded)
        HIP_TRY(hipStreamWaitEvent(cx->stream, g.noalloc_done, 0), "wait for the scratch array", layer);
    rc = decode_locked(n, kv, layer, seq_k, q_dev, out_dev, nq, scale_override, window, fixed);
    if (hipEventRecord(g.noalloc_done, cx->stream) == hipSuccess) g.noalloc_recorded = true;
    return rc;
}

int wr_hip_attn_append_decode_batched_dev(uint32_t n, wr_hip_kv* const* kv, uint32_t layer,
                                          const uint32_t* pos, const float* qkv_dev, uint32_t ld,
                                          uint32_t nq, const float* q_norm_dev, const float* k_norm_dev,
                                          float eps, const float* cos_sin_dev, uint32_t n_rot,
                                          float* out_dev, float scale_override, uint32_t window)
{
    if (!g.inited) return WR_HIP_ERR_STATE;
    if (!kv || !pos || !qkv_dev || !out_dev) return WR_HIP_ERR_INVAL;
    if (n == 0 || n > WR_HIP_BATCH_MAX) return WR_HIP_ERR_LIMIT;
    for (uint32_t i = 0; i < n; i++) {
        if (!kv[i]) return WR_HIP_ERR_INVAL;
        int rc = check_layer(kv[i], layer);
        if (rc) return rc;
    }
    const uint32_t hd = kv[0]->hd[layer], nkv = kv[0]->nkv;
    if (nq == 0 || nq % nkv != 0) return WR_HIP_ERR_INVAL;
    if ((q_norm_dev == nullptr) != (k_norm_dev == nullptr)) return WR_HIP_ERR_INVAL;
    if (n_rot > hd / 2 || (n_rot > 0 && !cos_sin_dev)) return WR_HIP_ERR_INVAL;
    if ((uint64_t)ld < (uint64_t)(nq + 2 * nkv) * hd) return WR_HIP_ERR_INVAL;
    // What the in-kernel form of the row step takes; for anything else the caller
    // keeps the two separate calls (nothing has been counted or written yet).
    const uintptr_t addrs = (uintptr_t)qkv_dev | (uintptr_t)cos_sin_dev | (uintptr_t)q_norm_dev |
                            (uintptr_t)k_norm_dev;
    if (hd != 128 || !mfma_shape(hd, nq / nkv) || n_rot % 8 != 0 || ld % 4 != 0 || addrs % 16 != 0)
        return WR_HIP_ERR_UNSUPPORTED;
    uint32_t seq_k[WR_HIP_BATCH_MAX];
    for (uint32_t i = 0; i < n; i++) {
        if (pos[i] >= kv[i]->max_ctx) return WR_HIP_ERR_CTX_FULL;          // as the append: nothing is written
        seq_k[i] = pos[i] + 1;
    }
    int rc = check_decode(n, kv, layer, seq_k, qkv_dev, out_dev, nq);      // the attention's own checks, the call counter
    if (rc) return rc;
    DecodeFusedArgs fz;
    memset(&fz, 0, sizeof fz);
    fz.qkv = qkv_dev;
    fz.q_norm = q_norm_dev;
    fz.k_norm = k_norm_dev;
    fz.cos_sin = n_rot ? cos_sin_dev : nullptr;
    fz.ld = ld;
    fz.n_rot = n_rot;
    fz.eps = eps;
    ENTER();
    return decode_locked(n, kv, layer, seq_k, nullptr, out_dev, nq, scale_override, window, DecodeWorkspace(), &fz);
}

// ------------------------------------------- a decode step's layers in one launch --

namespace {

constexpr uint32_t kStepRefusedSteps = 1000;   // steps that take the chain of launches after a wait has met its deadline

// Inputs and outputs of a product that a wave's registers hold a quarter of, four waves to the inputs (the rule
// of proj_chunk_locked), a tile (pair) to a workgroup.
bool step_product_ok(const wr_hip_weight* w, uint32_t n_in, uint32_t n_out, bool gated)
{
    if (!w || w->n_in != n_in || w->n_out != n_out) return false;
    const uint32_t tiles = n_out / 16, per_wave = n_in / 128;      // k-steps; in fours
    return n_in % 512 == 0 && per_wave <= kStepTiles / (gated ? 2 : 1) && tiles * 2 < 2048 &&
           tiles / (gated ? 2 : 1) <= g.n_cus;
}

// Whether another thread's work is under way that a step in one launch would keep waiting.  The launch holds
// every compute unit for its half millisecond, where a chain of small launches shares the device with other chains and
// with a prompt's launches.  28 layers, hidden 1024, threads that step a session of their own, us of all of them
// together per step, one launch at a time among them / chains: 2 threads 564 / 504, 3 560 / 380, 4 420 to 540 / 481, 5 474 /
// 415, 6 446 / 376 (8 375 / 397, 12 352 / 374).  A step beside prompts of 1024 tokens 1200 / 3100, the prompt 9000 /
// 6270; chains were all there was before, at 2700 and 6900.  Products of 2 to 16 rows fill the device as well and
// chains gain nothing beside them (steps beside steps of eight sessions, either 1560 / 1835): those do not count.
bool step_beside_others()
{
    std::lock_guard<std::mutex> lk(g.mu);
    for (const Ctx* c : g.ctxs) {
        const uint32_t rows = c->rows.load(std::memory_order_relaxed);
        if (c != cx && c->depth.load(std::memory_order_relaxed) && (rows < 2 || rows > WR_HIP_BATCH_MAX)) return true;
    }
    return false;
}

size_t step_part_bytes(uint32_t nq) { return (size_t)nq * kMergeInRegs * (128 + 2) * sizeof(uint64_t); }

}  // namespace

int wr_hip_attn_step_create(uint32_t n_layers, const wr_hip_attn_step_layer* layers, uint32_t nq, uint32_t nkv, uint32_t hd,
                            float eps, wr_hip_attn_step** out)
{
    if (!out) return WR_HIP_ERR_INVAL;
    *out = nullptr;
    if (!g.inited) return WR_HIP_ERR_STATE;
    if (n_layers == 0 || !layers || nq == 0 || nkv == 0 || nq % nkv != 0) return WR_HIP_ERR_INVAL;
    if (n_layers > WR_HIP_MAX_LAYERS) return WR_HIP_ERR_LIMIT;
    for (uint32_t l = 0; l < n_layers; l++) {
        const wr_hip_attn_step_layer& y = layers[l];
        if (!y.wqkv || !y.wo || !y.wgu || !y.wdown || !y.attn_norm || !y.ffn_norm) return WR_HIP_ERR_INVAL;
        if ((y.q_norm == nullptr) != (y.k_norm == nullptr)) return WR_HIP_ERR_INVAL;
    }
    const uint32_t hidden = layers[0].wqkv->n_in, ffn = layers[0].wdown->n_in;
    if (hd != 128 || nq / nkv > (uint32_t)kMaxGroupMfma || nq > kMaxHeads) return WR_HIP_ERR_UNSUPPORTED;
    StepLayer host[WR_HIP_MAX_LAYERS];
    for (uint32_t l = 0; l < n_layers; l++) {
        const wr_hip_attn_step_layer& y = layers[l];
        const uintptr_t addrs = (uintptr_t)y.attn_norm | (uintptr_t)y.ffn_norm | (uintptr_t)y.q_norm | (uintptr_t)y.k_norm;
        if (addrs % 16 != 0 || !step_product_ok(y.wqkv, hidden, (nq + 2 * nkv) * hd, false) ||
            !step_product_ok(y.wo, nq * hd, hidden, false) || !step_product_ok(y.wgu, hidden, 2 * ffn, true) ||
            !step_product_ok(y.wdown, ffn, hidden, false))
            return WR_HIP_ERR_UNSUPPORTED;
        host[l] = StepLayer{reinterpret_cast<const half8*>(y.wqkv->tiles), reinterpret_cast<const half8*>(y.wo->tiles),
                            reinterpret_cast<const half8*>(y.wgu->tiles), reinterpret_cast<const half8*>(y.wdown->tiles),
                            y.attn_norm, y.ffn_norm, y.q_norm, y.k_norm};
    }
    wr_hip_attn_step* p = new (std::nothrow) wr_hip_attn_step();
    if (!p) return WR_HIP_ERR_NOMEM;
    p->n_layers = n_layers;
    p->hidden = hidden;
    p->ffn = ffn;
    p->nq = nq;
    p->nkv = nkv;
    p->eps = eps;
    p->next_tag = 2;                     // (a cleared row bears tag 0, the row ahead of the first layer is not tagged)
    p->row_bytes = (size_t)(kStepCopies * (2 * step_row_units(hidden) + step_row_units(nq * hd) + step_row_units(ffn)) +
                            step_row_units((nq + 2 * nkv) * hd)) * 16 + step_part_bytes(nq);
    Entered entered_;
    int rc = entered_.ok() ? WR_HIP_OK : WR_HIP_ERR_NOMEM;
    if (rc == WR_HIP_OK && (device_malloc((void**)&p->layers, n_layers * sizeof(StepLayer)) != hipSuccess ||
                            device_malloc((void**)&p->rows, p->row_bytes) != hipSuccess))
        rc = WR_HIP_ERR_NOMEM;
    if (rc == WR_HIP_OK) {
        hipError_t e = hipMemcpyAsync(p->layers, host, n_layers * sizeof(StepLayer), hipMemcpyHostToDevice, cx->stream);
        if (e == hipSuccess) e = hipMemsetAsync(p->rows, 0, p->row_bytes, cx->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(cx->stream);
        if (e != hipSuccess) rc = hip_fail(e, "step plan", 0);
    }
    if (rc != WR_HIP_OK) {
        (void)hipGetLastError();
        wr_hip_attn_step_destroy(p);
        return rc;
    }
    *out = p;
    return WR_HIP_OK;
}

void wr_hip_attn_step_destroy(wr_hip_attn_step* p)
{
    if (!p) return;
    if (g.inited) {
        Entered entered_;
        if (entered_.ok()) (void)hipStreamSynchronize(cx->stream);
        if (p->layers) (void)hipFree(p->layers);
        if (p->rows) (void)hipFree(p->rows);
    }
    delete p;
}

void wr_hip_attn_set_alloc_failures(uint32_t n, uint32_t after)
{
    g.fail_after = after;
    g.fail_allocs = n;
}

void wr_hip_attn_step_set_tag(wr_hip_attn_step* p, uint32_t tag)
{
    if (p && tag >= 2) p->next_tag = tag;
}

void wr_hip_attn_set_step_limit(uint32_t ticks)
{
    g.step_limit = ticks;
    g.step_refused = 0;
}

int wr_hip_attn_step_dev(wr_hip_attn_step* p, wr_hip_kv* kv, uint32_t pos, float* row_dev, const float* cos_sin_dev,
                         uint32_t n_rot, float scale_override)
{
    if (!g.inited) return WR_HIP_ERR_STATE;
    if (!p || !kv || !row_dev || (n_rot > 0 && !cos_sin_dev) || n_rot > 64) return WR_HIP_ERR_INVAL;
    if (kv->n_layers != p->n_layers || kv->nkv != p->nkv) return WR_HIP_ERR_INVAL;
    for (uint32_t l = 0; l < kv->n_layers; l++)
        if (kv->hd[l] != 128) return WR_HIP_ERR_INVAL;
    if (pos >= kv->max_ctx) return WR_HIP_ERR_CTX_FULL;
    if (n_rot % 8 != 0 || (((uintptr_t)row_dev | (uintptr_t)cos_sin_dev) & 15) || !mfma_shape(128, p->nq / p->nkv))
        return WR_HIP_ERR_UNSUPPORTED;
    const uint32_t tiles = (pos + kTileKeys) / kTileKeys;
    const SplitRule r = split_rule(tiles, 128, true, g.tune_keys_per_wg.load(std::memory_order_relaxed));
    if (r.n_splits > (uint32_t)kMergeInRegs || p->nkv * r.n_splits > g.n_cus) return WR_HIP_ERR_UNSUPPORTED;
    ENTER();
    // A launch that is recorded would run again with the same tags.
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(cx->stream, &capture) != hipSuccess || capture != hipStreamCaptureStatusNone) {
        (void)hipGetLastError();
        return WR_HIP_ERR_UNSUPPORTED;
    }
    if (count_down(g.step_refused) || step_beside_others()) return WR_HIP_ERR_UNSUPPORTED;
    // Two launches whose workgroups wait for each other could each hold CUs the other needs: one at a time.
    Ctx* nobody = nullptr;
    if (!g.step_owner.compare_exchange_strong(nobody, cx, std::memory_order_acq_rel) && nobody != cx) return WR_HIP_ERR_UNSUPPORTED;

    if (p->next_tag > 0xFFFFFFFFu - 2 * p->n_layers) {
        // Tags begin again: what the rows still hold must not look like one to come.
        const uint32_t words = (uint32_t)(p->row_bytes / 4);
        hipLaunchKernelGGL(fill_u32_kernel, dim3((words + 255) / 256), dim3(256), 0, cx->stream, reinterpret_cast<uint32_t*>(p->rows), words, 0u);
        p->next_tag = 2;
    }
    StepArgs a;
    memset(&a, 0, sizeof a);
    a.layers = p->layers;
    a.x0 = row_dev;
    a.y = row_dev;
    a.cos_sin = n_rot ? cos_sin_dev : nullptr;
    kv->writes((uint64_t)pos + 1);
    a.slab = kv->slab;
    a.side = kv->vt_off[0];
    u32x4* at = p->rows;
    const auto take = [&](uint32_t n, uint32_t copies) { u32x4* row = at; at += copies * step_row_units(n); return row; };
    a.x = take(p->hidden, kStepCopies);
    a.x2 = take(p->hidden, kStepCopies);
    a.qkv = take((p->nq + 2 * p->nkv) * 128, 1);
    a.attn = take(p->nq * 128, kStepCopies);
    a.act = take(p->ffn, kStepCopies);
    a.part = reinterpret_cast<uint64_t*>(at);
    a.part_ml = a.part + (size_t)p->nq * kMergeInRegs * 128;
    a.expired = cx->err_dev + 1;
    a.s.seq_k = pos + 1;
    a.s.ctx_pad = kv->ctx_pad;
    a.s.n_splits = r.n_splits;
    a.s.tiles_per_wg = r.tiles_per_wg;
    a.s.tail_tiles = (uint16_t)r.tail;
    a.s.parts_per_wg = 1;
    a.n_layers = p->n_layers;
    a.hidden = p->hidden;
    a.ffn = p->ffn;
    a.nq = p->nq;
    a.nkv = p->nkv;
    a.n_rot = n_rot;
    a.tag0 = p->next_tag;
    const uint32_t limit = g.step_limit.load(std::memory_order_relaxed);
    a.limit = limit ? limit : kStepLimitTicks;
    a.eps = p->eps;
    a.qscale = (scale_override > 0.0f ? scale_override : 1.0f / sqrtf(128.0f)) * kLog2e;
    p->next_tag += p->n_layers;
    g.calls.fetch_add(p->n_layers, std::memory_order_relaxed);
    cx->step_calls = p->n_layers;
    const size_t lds = (size_t)kStepTiles * 128 * 4;       // terms of the most inputs
    launch_main(step_layers_kernel, dim3(g.n_cus), dim3(kStepThreads), a, lds);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        g.step_owner.store(nullptr, std::memory_order_release);
        return hip_fail(e, "step launch", 0);
    }
    return WR_HIP_OK;
}

int wr_hip_attn_step_done(void)
{
    if (!g.inited) return WR_HIP_ERR_STATE;
    ENTER();
    const int rc = sync_checked("step", 0);
    const bool late = cx->err_host[1] != 0;
    cx->err_host[1] = 0;
    Ctx* mine = cx;
    g.step_owner.compare_exchange_strong(mine, nullptr, std::memory_order_acq_rel);
    if (rc) return rc;
    if (late) {
        g.step_refused = kStepRefusedSteps;
        g.calls.fetch_sub(cx->step_calls, std::memory_order_relaxed);      // the step that is made instead counts its own
        return WR_HIP_ERR_STATE;
    }
    return WR_HIP_OK;
}

int wr_hip_attn_decode_batched(uint32_t n, wr_hip_kv* const* kv, uint32_t layer,
                               const uint32_t* seq_k, const float* const* q, float* const* out,
                               uint32_t nq, float scale_override, uint32_t window)
{
    int rc = check_decode(n, kv, layer, seq_k, q, out, nq);
    if (rc) return rc;
    for (uint32_t i = 0; i < n; i++)
        if (!q[i] || !out[i]) return WR_HIP_ERR_INVAL;
    const size_t row = (size_t)nq * kv[0]->hd[layer] * sizeof(float);
    ENTER();
    rc = ensure_device(cx->d_stage, 2 * n * row);
    if (rc) return rc;
    rc = ensure_pinned(cx->h_pin, n * row);
    if (rc) return rc;
    float* dq = reinterpret_cast<float*>(cx->d_stage.p);
    float* dout = reinterpret_cast<float*>((uint8_t*)cx->d_stage.p + n * row);
    for (uint32_t i = 0; i < n; i++) memcpy((uint8_t*)cx->h_pin.p + i * row, q[i], row);
    HIP_TRY(hipMemcpyAsync(dq, cx->h_pin.p, n * row, hipMemcpyHostToDevice, cx->stream), "q h2d",
            layer);
    rc = decode_locked(n, kv, layer, seq_k, dq, dout, nq, scale_override, window);
    if (rc) return rc;
    HIP_TRY(hipMemcpyAsync(cx->h_pin.p, dout, n * row, hipMemcpyDeviceToHost, cx->stream), "out d2h",
            layer);
    rc = sync_checked("decode sync", layer);
    if (rc) return rc;
    for (uint32_t i = 0; i < n; i++) memcpy(out[i], (uint8_t*)cx->h_pin.p + i * row, row);
    return WR_HIP_OK;
}

int wr_hip_attn_decode(wr_hip_kv* kv, uint32_t layer, uint32_t seq_k, const float* q, float* out,
                       uint32_t nq, float scale_override, uint32_t window)
{
    wr_hip_kv* kvs[1] = {kv};
    const float* qs[1] = {q};
    float* outs[1] = {out};
    if (!kv || !q || !out) return g.inited ? WR_HIP_ERR_INVAL : WR_HIP_ERR_STATE;
    return wr_hip_attn_decode_batched(1, kvs, layer, &seq_k, qs, outs, nq, scale_override, window);
}

int wr_hip_attn_append_decode_batched(uint32_t n, wr_hip_kv* const* kv, uint32_t layer,
                                      const uint32_t* pos, const float* const* k_f32,
                                      const float* const* v_f32, const float* const* q,
                                      float* const* out, uint32_t nq, float scale_override,
                                      uint32_t window)
{
    if (!g.inited) return WR_HIP_ERR_STATE;
    if (!kv || !pos || !k_f32 || !v_f32 || !q || !out) return WR_HIP_ERR_INVAL;
    if (n == 0 || n > WR_HIP_BATCH_MAX) return WR_HIP_ERR_LIMIT;
    for (uint32_t i = 0; i < n; i++) {
        if (!k_f32[i] || !v_f32[i] || !q[i] || !out[i]) return WR_HIP_ERR_INVAL;
        int rc = check_layer(kv[i], layer);
        if (rc) return rc;
    }
    const uint32_t hd = kv[0]->hd[layer], nkv = kv[0]->nkv;
    if (nq == 0 || nq % nkv != 0) return WR_HIP_ERR_INVAL;
    uint32_t seq_k[WR_HIP_BATCH_MAX];
    for (uint32_t i = 0; i < n; i++) {
        if (pos[i] >= kv[i]->max_ctx) return WR_HIP_ERR_CTX_FULL;          // as the append: nothing is written
        seq_k[i] = pos[i] + 1;
    }
    int rc = check_decode(n, kv, layer, seq_k, q, out, nq);
    if (rc) return rc;
    // One staged image, one copy up, the output rows behind it.  For the one-launch
    // kernel session i's rows lie as [nq Q | nkv K | nkv V], the stacked-projection
    // form it reads; for the two-step form the Q rows are packed in front (what the
    // attention reads) and the [K | V] pairs follow.
    const size_t qrow = (size_t)nq * hd, krow = (size_t)nkv * hd;
    const uint32_t ld = (uint32_t)(qrow + 2 * krow);
    const bool one_launch = hd == 128 && mfma_shape(hd, nq / nkv);
    const size_t in_bytes = (size_t)n * ld * sizeof(float), out_bytes = n * qrow * sizeof(float);
    ENTER();
    rc = ensure_device(cx->d_stage, in_bytes + out_bytes);
    if (rc) return rc;
    rc = ensure_pinned(cx->h_pin, in_bytes);
    if (rc) return rc;
    float* din = reinterpret_cast<float*>(cx->d_stage.p);
    float* dout = reinterpret_cast<float*>((uint8_t*)cx->d_stage.p + in_bytes);
    float* pin = reinterpret_cast<float*>(cx->h_pin.p);
    for (uint32_t i = 0; i < n; i++) {
        float* qdst = one_launch ? pin + (size_t)i * ld : pin + (size_t)i * qrow;
        float* kdst = one_launch ? qdst + qrow : pin + (size_t)n * qrow + (size_t)i * 2 * krow;
        memcpy(qdst, q[i], qrow * sizeof(float));
        memcpy(kdst, k_f32[i], krow * sizeof(float));
        memcpy(kdst + krow, v_f32[i], krow * sizeof(float));
    }
    HIP_TRY(hipMemcpyAsync(din, pin, in_bytes, hipMemcpyHostToDevice, cx->stream), "rows h2d", layer);
    if (one_launch) {
        // rows taken as they stand: no norm weights, no rotation
        DecodeFusedArgs fz;
        memset(&fz, 0, sizeof fz);
        fz.qkv = din;
        fz.ld = ld;
        rc = decode_locked(n, kv, layer, seq_k, nullptr, dout, nq, scale_override, window,
                           DecodeWorkspace(), &fz);
    } else {
        // the same two steps as separate launches on the one stream, no wait between them
        const float* dkv = din + (size_t)n * qrow;
        for (uint32_t i = 0; i < n && rc == WR_HIP_OK; i++)
            rc = append_rows_locked<float>(kv[i], layer, pos[i], 1, dkv + (size_t)i * 2 * krow,
                                           dkv + (size_t)i * 2 * krow + krow);
        if (rc == WR_HIP_OK)
            rc = decode_locked(n, kv, layer, seq_k, din, dout, nq, scale_override, window);
    }
    if (rc) return rc;
    HIP_TRY(hipMemcpyAsync(cx->h_pin.p, dout, out_bytes, hipMemcpyDeviceToHost, cx->stream), "out d2h",
            layer);
    rc = sync_checked("append+decode sync", layer);
    if (rc) return rc;
    for (uint32_t i = 0; i < n; i++)
        memcpy(out[i], (uint8_t*)cx->h_pin.p + i * qrow * sizeof(float), qrow * sizeof(float));
    return WR_HIP_OK;
}

int wr_hip_attn_append_decode(wr_hip_kv* kv, uint32_t layer, uint32_t pos, const float* k_f32,
                              const float* v_f32, const float* q, float* out, uint32_t nq,
                              float scale_override, uint32_t window)
{
    wr_hip_kv* kvs[1] = {kv};
    const float* ks[1] = {k_f32};
    const float* vs[1] = {v_f32};
    const float* qs[1] = {q};
    float* outs[1] = {out};
    return wr_hip_attn_append_decode_batched(1, kvs, layer, &pos, ks, vs, qs, outs, nq, scale_override,
                                             window);
}

// ---------------------------------------------------------------- prefill --

int wr_hip_attn_prefill_dev(wr_hip_kv* kv, uint32_t layer, uint32_t p0, uint32_t T,
                            const float* q_dev, float* out_dev, uint32_t nq, float scale_override,
                            uint32_t window)
{
    int rc = check_prefill(kv, layer, p0, T, q_dev, out_dev, nq);
    if (rc) return rc;
    ENTER();
    return prefill_locked(kv, layer, p0, T, q_dev, out_dev, nq, scale_override, window);
}

int wr_hip_attn_prefill_q16_dev(wr_hip_kv* kv, uint32_t layer, uint32_t p0, uint32_t T,
                                const uint16_t* q16_dev, float* out_dev, uint32_t nq, float scale_override,
                                uint32_t window)
{
    int rc = check_prefill(kv, layer, p0, T, q16_dev, out_dev, nq);
    if (rc) return rc;
    if (((uintptr_t)q16_dev & 7) != 0) return WR_HIP_ERR_INVAL;
    ENTER();
    return prefill_locked(kv, layer, p0, T, nullptr, out_dev, nq, scale_override, window, q16_dev);
}

int wr_hip_attn_prefill(wr_hip_kv* kv, uint32_t layer, uint32_t p0, uint32_t T, const float* q,
                        float* out, uint32_t nq, float scale_override, uint32_t window)
{
    int rc = check_prefill(kv, layer, p0, T, q, out, nq);
    if (rc) return rc;
    const size_t bytes = (size_t)T * nq * kv->hd[layer] * sizeof(float);
    ENTER();
    rc = ensure_device(cx->d_stage, 2 * bytes);
    if (rc) return rc;
    float* dq = reinterpret_cast<float*>(cx->d_stage.p);
    float* dout = reinterpret_cast<float*>((uint8_t*)cx->d_stage.p + bytes);
    rc = copy_up(dq, q, bytes, 0);
    if (rc == WR_HIP_OK)
        rc = prefill_locked(kv, layer, p0, T, dq, dout, nq, scale_override, window);
    if (rc == WR_HIP_OK) rc = copy_down_sync(out, dout, bytes);
    return rc;
}

// ------------------------------------------------------- device utilities --

void* wr_hip_attn_dev_alloc(size_t bytes)
{
    if (!g.inited || bytes == 0) return nullptr;
    Entered entered_;
    if (!entered_.ok()) return nullptr;
    void* p = nullptr;
    if (device_malloc(&p, bytes) != hipSuccess) return nullptr;
    return p;
}

void wr_hip_attn_dev_free(void* p)
{
    if (!g.inited || !p) return;
    Entered entered_;
    if (!entered_.ok()) return;
    (void)hipStreamSynchronize(cx->stream);
    (void)hipFree(p);
}

void* wr_hip_attn_host_alloc(size_t bytes)
{
    if (!g.inited || bytes == 0) return nullptr;
    Entered entered_;
    if (!entered_.ok()) return nullptr;
    void* p = nullptr;
    if (host_malloc(&p, bytes) != hipSuccess) return nullptr;
    return p;
}

void wr_hip_attn_host_free(void* p)
{
    if (!g.inited || !p) return;
    Entered entered_;
    if (!entered_.ok()) return;
    (void)hipStreamSynchronize(cx->stream);
    (void)hipHostFree(p);
}

int wr_hip_attn_h2d(void* dst_dev, const void* src_host, size_t bytes)
{
    if (!g.inited) return WR_HIP_ERR_STATE;
    if (!dst_dev || !src_host) return WR_HIP_ERR_INVAL;
    ENTER();
    HIP_TRY(hipMemcpyAsync(dst_dev, src_host, bytes, hipMemcpyHostToDevice, cx->stream), "h2d", 0);
    HIP_TRY(hipStreamSynchronize(cx->stream), "h2d sync", 0);
    return WR_HIP_OK;
}

int wr_hip_attn_d2h(void* dst_host, const void* src_dev, size_t bytes)
{
    if (!g.inited) return WR_HIP_ERR_STATE;
    if (!dst_host || !src_dev) return WR_HIP_ERR_INVAL;
    ENTER();
    HIP_TRY(hipMemcpyAsync(dst_host, src_dev, bytes, hipMemcpyDeviceToHost, cx->stream), "d2h", 0);
    return sync_checked("d2h sync", 0);
}

int wr_hip_attn_rows_d2h(uint32_t n, float* const* dst_locked, const float* src_dev, size_t row_floats)
{
    if (!g.inited) return WR_HIP_ERR_STATE;
    if (!dst_locked || !src_dev) return WR_HIP_ERR_INVAL;
    if (n == 0 || n > WR_HIP_BATCH_MAX) return WR_HIP_ERR_LIMIT;
    if (row_floats == 0 || row_floats % 4 != 0 || row_floats / 4 > 0x7FFFFFFFu || ((uintptr_t)src_dev & 15)) return WR_HIP_ERR_INVAL;
    RowsDownArgs a{};
    for (uint32_t i = 0; i < n; i++) {
        if (!dst_locked[i] || ((uintptr_t)dst_locked[i] & 15)) return WR_HIP_ERR_INVAL;
        a.dst[i] = reinterpret_cast<f32x4*>(dst_locked[i]);
    }
    a.src = reinterpret_cast<const f32x4*>(src_dev);
    a.units = a.ld_units = (uint32_t)(row_floats / 4);
    ENTER();
    hipLaunchKernelGGL(rows_down_kernel, dim3(std::min((a.units + 255) / 256, 64u), n), dim3(256), 0, cx->stream, a);
    HIP_TRY(hipGetLastError(), "rows down launch", 0);
    return sync_checked("rows down", 0);
}

int wr_hip_attn_sync(void)
{
    if (!g.inited) return WR_HIP_ERR_STATE;
    ENTER();
    return sync_checked("sync", 0);
}

void* wr_hip_attn_stream(void)
{
    Entered entered_;
    return entered_.ok() ? (void*)cx->stream : nullptr;
}

// ------------------------------------------------------------ projections --

int wr_hip_proj_weight_create(uint32_t n_parts, const uint16_t* const* parts_f16,
                              const uint32_t* rows_per_part, uint32_t n_in, wr_hip_weight** out)
{
    if (!out) return WR_HIP_ERR_INVAL;
    *out = nullptr;
    if (!g.inited) return WR_HIP_ERR_STATE;
    if (n_parts == 0 || !parts_f16 || !rows_per_part || n_in == 0 || n_in % 32 != 0)
        return WR_HIP_ERR_INVAL;
    uint64_t n_out = 0;
    for (uint32_t i = 0; i < n_parts; i++) {
        if (!parts_f16[i] || rows_per_part[i] == 0) return WR_HIP_ERR_INVAL;
        n_out += rows_per_part[i];
    }
    if (n_out % 16 != 0 || n_out > 0x7FFFFFFFu) return WR_HIP_ERR_INVAL;
    wr_hip_weight* w = new (std::nothrow) wr_hip_weight();
    if (!w) return WR_HIP_ERR_NOMEM;
    w->n_out = (uint32_t)n_out;
    w->n_in = n_in;
    w->bytes = (size_t)n_out * n_in * 2;
    w->tiles = nullptr;

    ENTER();
    void* rowmajor = nullptr;
    hipError_t e = device_malloc((void**)&w->tiles, w->bytes);
    if (e == hipSuccess) e = device_malloc((void**)&rowmajor, w->bytes);
    if (e != hipSuccess) {
        logmsg(0, "projection: device weight alloc failed (%zu bytes): %s", w->bytes,
               hipGetErrorString(e));
        if (w->tiles) (void)hipFree(w->tiles);
        delete w;
        return WR_HIP_ERR_NOMEM;
    }
    size_t off = 0;
    for (uint32_t i = 0; i < n_parts && e == hipSuccess; i++) {
        const size_t nb = (size_t)rows_per_part[i] * n_in * 2;
        e = hipMemcpyAsync((uint8_t*)rowmajor + off, parts_f16[i], nb, hipMemcpyHostToDevice, cx->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(cx->stream);     // pageable source
        off += nb;
    }
    if (e == hipSuccess) {
        const size_t units = w->bytes / 16;
        hipLaunchKernelGGL(proj_pack_weights_kernel, dim3((uint32_t)((units + 255) / 256)), dim3(256),
                           0, cx->stream, reinterpret_cast<const uint16_t*>(rowmajor),
                           reinterpret_cast<u32x4*>(w->tiles), w->n_out, w->n_in);
        e = hipGetLastError();
        if (e == hipSuccess) e = hipStreamSynchronize(cx->stream);
    }
    (void)hipFree(rowmajor);
    if (e != hipSuccess) {
        (void)hipFree(w->tiles);
        delete w;
        return hip_fail(e, "weight upload", 0);
    }
    *out = w;
    return WR_HIP_OK;
}

void wr_hip_proj_weight_destroy(wr_hip_weight* w)
{
    if (!w) return;
    if (g.inited) {
        Entered entered_;
        if (entered_.ok()) (void)hipStreamSynchronize(cx->stream);
        (void)hipFree(w->tiles);
    }
    delete w;
}

static int check_proj(const wr_hip_weight* w, uint32_t rows, const void* x, uint32_t ldx,
                      uint32_t min_ldx, const void* y, uint32_t ldy, uint32_t min_ldy)
{
    if (!g.inited) return WR_HIP_ERR_STATE;
    if (!w || !x || !y) return WR_HIP_ERR_INVAL;
    if (rows == 0) return WR_HIP_OK;
    if (ldx < min_ldx || ldy < min_ldy || ldy % 4 != 0) return WR_HIP_ERR_INVAL;
    return WR_HIP_OK;
}

static int proj_dev_common(const wr_hip_weight* w, uint32_t rows, const float* x_dev, uint32_t ldx,
                           uint32_t min_ldx, const ProjSource& src, const float* add_dev,
                           float* y_dev, uint32_t ldy)
{
    int rc = check_proj(w, rows, x_dev, ldx, min_ldx, y_dev, ldy, w ? w->n_out : 0);
    if (rc || rows == 0) return rc;
    if (((uintptr_t)y_dev & 15) || (add_dev && ((uintptr_t)add_dev & 15))) return WR_HIP_ERR_INVAL;
    ENTER();
    return proj_locked(w, rows, x_dev, ldx, src, add_dev, y_dev, ldy);
}

int wr_hip_proj_rows_dev(const wr_hip_weight* w, uint32_t rows, const float* x_dev, uint32_t ldx,
                         const float* add_dev, float* y_dev, uint32_t ldy)
{
    return proj_dev_common(w, rows, x_dev, ldx, w ? w->n_in : 0, ProjSource(), add_dev, y_dev, ldy);
}

int wr_hip_proj_rows_norm_dev(const wr_hip_weight* w, uint32_t rows, const float* x_dev,
                              uint32_t ldx, const float* norm_w_dev, float eps,
                              const float* add_dev, float* y_dev, uint32_t ldy)
{
    if (g.inited && !norm_w_dev) return WR_HIP_ERR_INVAL;
    ProjSource src;
    src.kind = kProjSrcRmsNorm;
    src.norm_w = norm_w_dev;
    src.eps = eps;
    return proj_dev_common(w, rows, x_dev, ldx, w ? w->n_in : 0, src, add_dev, y_dev, ldy);
}

int wr_hip_proj_rows_norm_down(const wr_hip_weight* w, uint32_t rows, const float* x_dev, uint32_t ldx,
                               const float* norm_w_dev, float eps, float* const* dst_locked, float* tmp_dev)
{
    int rc = check_proj(w, rows, x_dev, ldx, w ? w->n_in : 0, dst_locked, w ? w->n_out : 0, w ? w->n_out : 0);
    if (rc || rows == 0) return rc;
    if (rows > WR_HIP_BATCH_MAX) return WR_HIP_ERR_LIMIT;
    if (!norm_w_dev || (rows > 1 && !tmp_dev) || ((uintptr_t)tmp_dev & 15)) return WR_HIP_ERR_INVAL;
    ProjDownArgs d{};
    for (uint32_t i = 0; i < rows; i++) {
        if (!dst_locked[i] || ((uintptr_t)dst_locked[i] & 15)) return WR_HIP_ERR_INVAL;
        d.y[i] = reinterpret_cast<f32x4*>(dst_locked[i]);
    }
    ProjSource src;
    src.kind = kProjSrcRmsNorm;
    src.norm_w = norm_w_dev;
    src.eps = eps;
    ENTER();
    if (rows > 1 && proj_ksplit(w) == 1) {
        rc = proj_chunk_locked(w, rows, x_dev, ldx, src, nullptr, tmp_dev, w->n_out, &d);
        return rc ? rc : sync_checked("product down", 0);
    }
    rc = proj_locked(w, rows, x_dev, ldx, src, nullptr, rows == 1 ? dst_locked[0] : tmp_dev, w->n_out);
    if (rc) return rc;
    return rows == 1 ? sync_checked("product down", 0) : wr_hip_attn_rows_d2h(rows, dst_locked, tmp_dev, w->n_out);
}

int wr_hip_proj_rows_swiglu_dev(const wr_hip_weight* w, uint32_t rows, const float* gate_up_dev,
                                uint32_t ld, const float* add_dev, float* y_dev, uint32_t ldy)
{
    ProjSource src;
    src.kind = kProjSrcSwiglu;
    return proj_dev_common(w, rows, gate_up_dev, ld, w ? 2 * w->n_in : 0, src, add_dev, y_dev, ldy);
}

int wr_hip_proj_rows_geglu_dev(const wr_hip_weight* w, uint32_t rows, const float* gate_up_dev,
                               uint32_t ld, const float* add_dev, float* y_dev, uint32_t ldy)
{
    ProjSource src;
    src.kind = kProjSrcGeglu;
    return proj_dev_common(w, rows, gate_up_dev, ld, w ? 2 * w->n_in : 0, src, add_dev, y_dev, ldy);
}

int wr_hip_proj_rows_gated_dev(const wr_hip_weight* w, uint32_t rows, const float* x_dev, uint32_t ldx,
                               const float* norm_w_dev, float eps, int gelu, float* act_dev, uint32_t ldo)
{
    if (w && w->n_out % 32) return WR_HIP_ERR_INVAL;
    int rc = check_proj(w, rows, x_dev, ldx, w ? w->n_in : 0, act_dev, ldo, w ? w->n_out / 2 : 0);
    if (rc || rows == 0) return rc;
    if ((uintptr_t)act_dev & 15) return WR_HIP_ERR_INVAL;
    ProjSource src;
    src.kind = norm_w_dev ? kProjSrcRmsNorm : kProjSrcPlain;
    src.norm_w = norm_w_dev;
    src.eps = eps;
    src.gate = gelu ? kProjSrcGeglu : kProjSrcSwiglu;
    ENTER();
    return proj_locked(w, rows, x_dev, ldx, src, nullptr, act_dev, ldo);
}

int wr_hip_proj_embed_dev(const wr_hip_weight* w, uint32_t rows, const uint32_t* tokens, float scale, float* x_dev, uint32_t ldx)
{
    int rc = check_proj(w, rows, tokens, 0, 0, x_dev, ldx, w ? w->n_in : 0);
    if (rc || rows == 0) return rc;
    if ((uintptr_t)x_dev & 15) return WR_HIP_ERR_INVAL;
    for (uint32_t r = 0; r < rows; r++)
        if (tokens[r] >= w->n_out) return WR_HIP_ERR_INVAL;               // never clamped
    ENTER();
    ProjEmbedArgs a;
    a.w = reinterpret_cast<const half8*>(w->tiles);
    a.ldx = ldx;
    a.K = w->n_in;
    a.scale = scale;
    for (uint32_t done = 0; done < rows; done += kEmbedTokens) {
        const uint32_t n = std::min(rows - done, kEmbedTokens);
        a.x = x_dev + (size_t)done * ldx;
        memcpy(a.tokens, tokens + done, n * sizeof(uint32_t));
        hipLaunchKernelGGL(proj_embed_kernel, dim3(n), dim3(128), 0, cx->stream, a);
    }
    HIP_TRY(hipGetLastError(), "embedding launch", 0);
    return WR_HIP_OK;
}

int wr_hip_proj_rows(const wr_hip_weight* w, uint32_t rows, const float* x, float* y)
{
    if (w && (w->n_out % 4 != 0)) return WR_HIP_ERR_INVAL;
    int rc = check_proj(w, rows, x, w ? w->n_in : 0, w ? w->n_in : 0, y, w ? w->n_out : 0, w ? w->n_out : 0);
    if (rc || rows == 0) return rc;
    const size_t xb = ((size_t)rows * w->n_in * sizeof(float) + 255) & ~(size_t)255;
    const size_t yb = (size_t)rows * w->n_out * sizeof(float);
    ENTER();
    rc = ensure_device(cx->d_stage, xb + yb);
    if (rc) return rc;
    float* dx = reinterpret_cast<float*>(cx->d_stage.p);
    float* dy = reinterpret_cast<float*>((uint8_t*)cx->d_stage.p + xb);
    rc = copy_up(dx, x, (size_t)rows * w->n_in * sizeof(float), 0);
    if (rc == WR_HIP_OK) rc = proj_locked(w, rows, dx, w->n_in, ProjSource(), nullptr, dy, w->n_out);
    if (rc == WR_HIP_OK) rc = copy_down_sync(y, dy, yb);
    return rc;
}

// ------------------------------------------------------------- row steps --

int wr_hip_rows_rmsnorm_dev(const float* x_dev, uint32_t ldx, const float* w_dev, uint32_t wn,
                            float* out_dev, uint32_t ldo, uint32_t rows, uint32_t dim, float eps)
{
    if (!g.inited) return WR_HIP_ERR_STATE;
    if (!x_dev || !out_dev || dim == 0 || ldx < dim || ldo < dim) return WR_HIP_ERR_INVAL;
    if (wn > 0 && !w_dev) return WR_HIP_ERR_INVAL;
    if (rows == 0) return WR_HIP_OK;
    ENTER();
    hipLaunchKernelGGL(rmsnorm_rows_kernel, dim3(rows), dim3(256), 0, cx->stream, x_dev, ldx, w_dev, wn,
                       out_dev, ldo, dim, eps, 0);
    HIP_TRY(hipGetLastError(), "rmsnorm launch", 0);
    return WR_HIP_OK;
}

int wr_hip_rows_rmsnorm_add_dev(const float* x_dev, uint32_t ldx, const float* w_dev, uint32_t wn,
                                float* acc_dev, uint32_t lda, uint32_t rows, uint32_t dim, float eps)
{
    if (!g.inited) return WR_HIP_ERR_STATE;
    if (!x_dev || !acc_dev || dim == 0 || ldx < dim || lda < dim) return WR_HIP_ERR_INVAL;
    if (wn > 0 && !w_dev) return WR_HIP_ERR_INVAL;
    if (rows == 0) return WR_HIP_OK;
    ENTER();
    hipLaunchKernelGGL(rmsnorm_rows_kernel, dim3(rows), dim3(256), 0, cx->stream, x_dev, ldx, w_dev, wn,
                       acc_dev, lda, dim, eps, 1);
    HIP_TRY(hipGetLastError(), "rmsnorm + add launch", 0);
    return WR_HIP_OK;
}

int wr_hip_rows_qkv_prep_dev(const float* qkv_dev, uint32_t ld, uint32_t rows, uint32_t nq,
                             uint32_t nkv, uint32_t hd, const float* q_norm_dev,
                             const float* k_norm_dev, float eps, const float* cos_sin_dev,
                             uint32_t n_rot, float* q_out_dev, float* k_out_dev, float* v_out_dev)
{
    if (!g.inited) return WR_HIP_ERR_STATE;
    if (!qkv_dev || !q_out_dev || !k_out_dev || !v_out_dev) return WR_HIP_ERR_INVAL;
    if (nq == 0 || nkv == 0 || hd < 2 || (hd & 1) || hd > (uint32_t)kRowsMaxHd) return WR_HIP_ERR_INVAL;
    if ((uint64_t)ld < (uint64_t)(nq + 2 * nkv) * hd) return WR_HIP_ERR_INVAL;
    if (n_rot > hd / 2 || (n_rot > 0 && !cos_sin_dev)) return WR_HIP_ERR_INVAL;
    if ((q_norm_dev == nullptr) != (k_norm_dev == nullptr)) return WR_HIP_ERR_INVAL;
    if (rows == 0) return WR_HIP_OK;
    QkvPrepArgs a;
    a.qkv = qkv_dev;
    a.q_norm = q_norm_dev;
    a.k_norm = k_norm_dev;
    a.cos_sin = cos_sin_dev;
    a.q_out = q_out_dev;
    a.k_out = k_out_dev;
    a.v_out = v_out_dev;
    a.ld = ld;
    a.nq = nq;
    a.nkv = nkv;
    a.hd = hd;
    a.n_rot = n_rot;
    a.eps = eps;
    ENTER();
    hipLaunchKernelGGL(qkv_prep_kernel, dim3(rows, nq + 2 * nkv), dim3(64), 0, cx->stream, a);
    HIP_TRY(hipGetLastError(), "qkv prep launch", 0);
    return WR_HIP_OK;
}

// q16_out_dev != nullptr: Q leaves as binary16 rows multiplied by the softmax
// scale times log2(e) (what wr_hip_attn_prefill_q16_dev takes) instead of F32.
static int qkv_append_common(const float* qkv_dev, uint32_t ld, uint32_t rows, uint32_t nq,
                             const float* q_norm_dev, const float* k_norm_dev, float eps,
                             const float* cos_sin_dev, uint32_t n_rot, uint32_t n_kv,
                             wr_hip_kv* const* kv, uint32_t layer, const uint32_t* pos,
                             float* q_out_dev, uint16_t* q16_out_dev, float scale_override, uint32_t flags)
{
    if (!g.inited) return WR_HIP_ERR_STATE;
    if (!qkv_dev || (!q_out_dev && !q16_out_dev) || !kv || !pos || nq == 0) return WR_HIP_ERR_INVAL;
    if (flags & ~(uint32_t)(WR_HIP_QKV_V_NORM | WR_HIP_QKV_Q_ONLY)) return WR_HIP_ERR_INVAL;
    const bool q_only = (flags & WR_HIP_QKV_Q_ONLY) != 0;
    if (n_kv == 0 || (n_kv != 1 && n_kv != rows)) return WR_HIP_ERR_INVAL;
    if (n_kv > WR_HIP_BATCH_MAX) return WR_HIP_ERR_LIMIT;
    QkvAppendArgs a;
    memset(&a, 0, sizeof a);
    for (uint32_t i = 0; i < n_kv; i++) {
        int rc = check_layer(kv[i], layer);
        if (rc) return rc;
        if (kv[i]->nkv != kv[0]->nkv || kv[i]->hd[layer] != kv[0]->hd[layer]) return WR_HIP_ERR_INVAL;
        for (uint32_t j = 0; j < i; j++)
            if (kv[i] == kv[j]) return WR_HIP_ERR_INVAL;
        const uint64_t end = (uint64_t)pos[i] + (n_kv == 1 ? rows : 1);
        if (!q_only && end > kv[i]->max_ctx) return WR_HIP_ERR_CTX_FULL;   // nothing is written
        a.k[i] = reinterpret_cast<uint16_t*>(kv[i]->slab + kv[i]->k_off[layer]);
        a.vt[i] = reinterpret_cast<uint16_t*>(kv[i]->slab + kv[i]->vt_off[layer]);
        a.pos[i] = pos[i];
        a.ctx_pad[i] = kv[i]->ctx_pad;
    }
    const uint32_t nkv = kv[0]->nkv, hd = kv[0]->hd[layer];
    if (hd < 2 || (hd & 1)) return WR_HIP_ERR_INVAL;
    if (hd > 512) return WR_HIP_ERR_LIMIT;                // the V block gathered in LDS: hd * 68 bytes
    if ((uint64_t)ld < (uint64_t)(nq + (q_only ? 0 : 2 * nkv)) * hd) return WR_HIP_ERR_INVAL;
    if (n_rot > hd / 2 || (n_rot > 0 && !cos_sin_dev)) return WR_HIP_ERR_INVAL;
    if (!q_only && (q_norm_dev == nullptr) != (k_norm_dev == nullptr)) return WR_HIP_ERR_INVAL;
    if (rows == 0) return WR_HIP_OK;
    a.v_norm = (flags & WR_HIP_QKV_V_NORM) ? 1 : 0;
    a.qkv = qkv_dev;
    a.q_norm = q_norm_dev;
    a.k_norm = k_norm_dev;
    a.cos_sin = n_rot ? cos_sin_dev : nullptr;           // a table of zero pairs per row holds nothing to read
    a.q_out = q_out_dev;
    a.ld = ld;
    a.nq = nq;
    a.nkv = nkv;
    a.hd = hd;
    a.n_rot = n_rot;
    a.rows = rows;
    a.per_session = (n_kv > 1 || rows == 1) ? 1 : 0;
    a.eps = eps;
    {
        // eight lanes per position with 16-byte accesses where the shapes and
        // the addresses allow it (every model on the device walk does)
        const uintptr_t addrs = (uintptr_t)qkv_dev | (uintptr_t)q_out_dev | (uintptr_t)q16_out_dev |
                                (uintptr_t)cos_sin_dev | (uintptr_t)q_norm_dev | (uintptr_t)k_norm_dev;
        if ((hd == 128 || hd == 256) && n_rot % 8 == 0 && ld % 4 == 0 && addrs % 16 == 0) a.row8 = hd / 64;
    }
    if (q16_out_dev) {
        // only the eight-lane form writes it, and only the 128-wide head has a
        // prefill kernel that reads it
        if (a.row8 != 2) return WR_HIP_ERR_UNSUPPORTED;
        const float scale = (scale_override > 0.0f) ? scale_override : 1.0f / sqrtf((float)hd);
        a.q16_out = q16_out_dev;
        a.q16_scale = scale * kLog2e;                     // prefill_locked's qscale, by the same expression
    }
    const uint32_t gx = a.per_session ? rows : (pos[0] + rows - 1) / kVBlock - pos[0] / kVBlock + 1;
    const size_t lds = std::max((size_t)4 * hd * sizeof(float), (size_t)hd * (kVBlock + 2) * sizeof(uint16_t));
    ENTER();
    if (!q_only)
        for (uint32_t i = 0; i < n_kv; i++) kv[i]->writes((uint64_t)pos[i] + (n_kv == 1 ? rows : 1));
    hipLaunchKernelGGL(qkv_append_kernel, dim3(gx, nq + (q_only ? 0 : 2 * nkv)), dim3(256), lds, cx->stream, a);
    HIP_TRY(hipGetLastError(), "qkv append launch", layer);
    return WR_HIP_OK;
}

int wr_hip_rows_qkv_append_dev(const float* qkv_dev, uint32_t ld, uint32_t rows, uint32_t nq,
                               const float* q_norm_dev, const float* k_norm_dev, float eps,
                               const float* cos_sin_dev, uint32_t n_rot, uint32_t n_kv,
                               wr_hip_kv* const* kv, uint32_t layer, const uint32_t* pos,
                               float* q_out_dev, uint32_t flags)
{
    if (!q_out_dev) return g.inited ? WR_HIP_ERR_INVAL : WR_HIP_ERR_STATE;
    return qkv_append_common(qkv_dev, ld, rows, nq, q_norm_dev, k_norm_dev, eps, cos_sin_dev, n_rot, n_kv, kv,
                             layer, pos, q_out_dev, nullptr, 0.0f, flags);
}

int wr_hip_rows_qkv_append_q16_dev(const float* qkv_dev, uint32_t ld, uint32_t rows, uint32_t nq,
                                   const float* q_norm_dev, const float* k_norm_dev, float eps,
                                   const float* cos_sin_dev, uint32_t n_rot, uint32_t n_kv,
                                   wr_hip_kv* const* kv, uint32_t layer, const uint32_t* pos,
                                   uint16_t* q16_out_dev, float scale_override, uint32_t flags)
{
    if (!q16_out_dev) return g.inited ? WR_HIP_ERR_INVAL : WR_HIP_ERR_STATE;
    return qkv_append_common(qkv_dev, ld, rows, nq, q_norm_dev, k_norm_dev, eps, cos_sin_dev, n_rot, n_kv, kv,
                             layer, pos, nullptr, q16_out_dev, scale_override, flags);
}

int wr_hip_rows_swiglu_dev(const float* gate_up_dev, uint32_t ld, float* act_dev, uint32_t ldo,
                           uint32_t rows, uint32_t ffn)
{
    if (!g.inited) return WR_HIP_ERR_STATE;
    if (!gate_up_dev || !act_dev || ffn == 0 || (uint64_t)ld < 2ull * ffn || ldo < ffn)
        return WR_HIP_ERR_INVAL;
    if (rows == 0) return WR_HIP_OK;
    ENTER();
    const size_t total = (size_t)rows * ffn;
    hipLaunchKernelGGL(swiglu_rows_kernel, dim3((uint32_t)((total + 255) / 256)), dim3(256), 0,
                       cx->stream, gate_up_dev, ld, act_dev, ldo, rows, ffn);
    HIP_TRY(hipGetLastError(), "swiglu launch", 0);
    return WR_HIP_OK;
}

uint32_t wr_hip_proj_weight_rows(const wr_hip_weight* w) { return w ? w->n_out : 0; }
uint32_t wr_hip_proj_weight_cols(const wr_hip_weight* w) { return w ? w->n_in : 0; }

int wr_hip_attn_profile_begin(uint32_t max_launches)
{
    if (!g.inited) return WR_HIP_ERR_STATE;
    ENTER();
    HIP_TRY(hipStreamSynchronize(cx->stream), "sync", 0);
    while (cx->ev.size() < 2 * (size_t)max_launches) {
        hipEvent_t e;
        HIP_TRY(hipEventCreate(&e), "event create", 0);
        cx->ev.push_back(e);
    }
    cx->ev_used = 0;
    cx->profiling = true;
    return WR_HIP_OK;
}

int wr_hip_attn_profile_end(double* total_ms, uint32_t* n_launches)
{
    if (!g.inited) return WR_HIP_ERR_STATE;
    ENTER();
    HIP_TRY(hipStreamSynchronize(cx->stream), "sync", 0);
    double sum = 0.0;
    for (uint32_t i = 0; i + 1 < cx->ev_used; i += 2) {
        float ms = 0.f;
        HIP_TRY(hipEventElapsedTime(&ms, cx->ev[i], cx->ev[i + 1]), "event elapsed", 0);
        sum += ms;
    }
    if (total_ms) *total_ms = sum;
    if (n_launches) *n_launches = cx->ev_used / 2;
    cx->profiling = false;
    cx->ev_used = 0;
    return WR_HIP_OK;
}

}  // extern "C"
