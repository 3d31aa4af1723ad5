// What the device library's translation units share: the library's state, the
// calling thread's context (stream, staging, tickets, error word), logging,
// copies and kernel launches.  Defined in wr_hip_attn.hip.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include <atomic>
#include <cstdint>
#include <mutex>
#include <vector>

#include "../../include/wr_hip_attn.h"

namespace wr {

constexpr int kMaxDevices = 16;
constexpr uint32_t kMaxPrefillParts = 32;    // prefill: parts a block's keys are cut into at most,
constexpr uint32_t kMaxPrefillPartMb = 128;  // and the MiB that the parts' rows take
constexpr uint32_t kRefusedLaunches = 1000;  // that do without optional memory before it is asked for again

struct Buffer {
    void* p = nullptr;
    size_t cap = 0;
};

// What one calling thread submits through: its own stream, so that sessions
// driven from different threads overlap on the device (the reference lets
// independent sessions run concurrently, include/wayruntime.h:29-40), and the
// buffers whose contents belong to the launches on that stream.
struct Ctx {
    hipStream_t stream = nullptr;
    Buffer d_stage;              // device staging for host-pointer entry points
    Buffer d_part;               // split-K partials
    Buffer d_picked;             // experts' rows in slot order: at most kMaxPickedBytes, none where it is refused
    uint32_t picked_refused = 0;      // launches that do without before memory for them is asked for again
    Buffer d_prefill;            // rows of prefill blocks cut into parts: at most kMaxPrefillPartMb, none where it is refused
    uint32_t prefill_refused = 0;     // launches that go uncut before memory for them is asked for again
    Buffer d_proj;               // projection operand fragments and row scales
    uint32_t* d_counters = nullptr;   // split-K tickets, zero whenever no launch is in flight
    // Error word: page-locked host memory that kernels can write.  A kernel that
    // gives up a bounded wait (and so goes on with data it cannot vouch for) stores
    // (bit 31 | layer) there; the host reads it after every wait for the
    // stream (no copy, no extra latency).  Nothing writes it today.  The word behind it is
    // step_layers_kernel's, whose waits are bounded: set when one met its deadline, and
    // read by wr_hip_attn_step_done, after which the step is made another way.
    volatile uint32_t* err_host = nullptr;
    uint32_t* err_dev = nullptr;
    // Read by other threads, to see whose work runs beside theirs: how deep the thread is in calls that touch the device
    // (one may make another), and how many rows its last product had.
    std::atomic<uint32_t> depth{0}, rows{0};
    uint32_t step_calls = 0;          // attention calls that the last step in one launch counted
    Buffer h_pin;                // pinned host staging
    std::vector<hipEvent_t> ev;  // kernel timing (profile_begin / profile_end of this thread)
    uint32_t ev_used = 0;
    bool profiling = false;
};

// Where a cache has been written (clear_cache_kernel).
struct ClearArgs {
    uint32_t nkv, ctx_pad, tiles;        // tiles: runs of 32 positions, from the first on
    uint32_t hd[WR_HIP_MAX_LAYERS];      // 0: no cache
    uint64_t k_off[WR_HIP_MAX_LAYERS], vt_off[WR_HIP_MAX_LAYERS];
};

struct Lib {
    std::mutex mu;               // init / shutdown, the set of thread contexts, the knobs
    std::atomic<bool> inited{false};   // read without the lock by every entry point
    int device = -1;
    uint32_t n_cus = 256;        // compute units of the device in use
    std::atomic<uint64_t> generation{0};   // bumped by every init: contexts of an earlier one are gone
    std::vector<Ctx*> ctxs;      // every context of this generation
    struct Slab {
        uint8_t* p;
        size_t bytes;
        uint32_t n_layers;
        ClearArgs cleared;       // where its last cache has written
    };
    std::mutex slab_mu;          // guards slabs; nothing else is locked while it is held
    std::vector<Slab> slabs;     // memory of ended caches; what they wrote is cleared when it is taken again
    std::vector<Ctx*> idle;      // contexts whose thread has ended, for the next new thread
    char name[320] = "uninitialised";
    unsigned char* noalloc_ws[kMaxDevices] = {};   // device address of `scratch`, per device
    // The fixed scratch array is one per device: launches that use it are
    // chained across threads' streams through this event (recorded after each,
    // waited for before the next), under its own lock.
    std::mutex noalloc_mu;
    hipEvent_t noalloc_done = nullptr;
    bool noalloc_recorded = false;
    std::atomic<uint64_t> calls{0};
    wr_hip_log_fn log_fn = nullptr;
    void* log_user = nullptr;
    std::atomic<uint32_t> tune_keys_per_wg{0};
    std::atomic<int> force_generic{0};
    std::atomic<uint32_t> prefill_part_mb{kMaxPrefillPartMb};    // WR_HIP_PREFILL_PART_MB: a thread's parts take no more; 0: no block is cut
    std::atomic<int> prefill_256_four_waves{0};   // WR_HIP_PREFILL_256_FOUR_WAVES=1: head dim 256 keeps the earlier four-wave prefill kernel
    std::atomic<Ctx*> step_owner{nullptr};       // whose launch of a whole step's layers may be on the device (one at a time)
    std::atomic<uint32_t> step_refused{0};       // steps that go layer by layer before one launch is tried again
    std::atomic<uint32_t> step_limit{0};         // ticks until its waits end; 0: kStepLimitTicks
    std::atomic<uint32_t> fail_allocs{0}, fail_after{0};   // for tests: this many allocations fail, behind so many that do not
    std::atomic<int> prefill_two_waves{1};        // WR_HIP_PREFILL_TWO_WAVES=0: head dim 128 takes the one-wave-per-SIMD prefill kernel
};
extern Lib g;

// The calling thread's context (set by Entered, below).
extern thread_local Ctx* cx;

constexpr uint32_t kDevErrLayerMask = 0x0000FFFFu;     // error word: bit 31 set (kDevErrWaitExpired), the layer in the low bits
constexpr float kLog2e = 1.4426950408889634f;
constexpr uint32_t kDefaultTilesPerWg = 32;  // split-K decode: 1024 keys per workgroup
constexpr uint32_t kMaxHeads = 4096;        // query heads per session the ticket array is sized for
constexpr size_t kOnePerCuLds = 82 * 1024;  // more than half of a compute unit's LDS
constexpr size_t kPinSmall = 1u << 20;      // host copies up to this size go through pinned staging

void logmsg(int level, const char* fmt, ...);
int hip_fail(hipError_t e, const char* what, uint32_t layer);

#define HIP_TRY(expr, what, layer)                                   \
    do {                                                             \
        hipError_t e_ = (expr);                                      \
        if (e_ != hipSuccess) return hip_fail(e_, what, layer);      \
    } while (0)

hipError_t device_malloc(void** p, size_t bytes);
int ensure_device(Buffer& b, size_t need);
int ensure_pinned(Buffer& b, size_t need);
bool optional_device(Buffer& b, uint32_t& refused, size_t need, const char* without);
int sync_checked(const char* what, uint32_t layer);
int copy_up(void* dst_dev, const void* src_host, size_t bytes, size_t pin_off);
int copy_down_sync(void* dst_host, const void* src_dev, size_t bytes);

template <typename Kern, typename A0, typename A1>
void launch_main(Kern kernel, dim3 grid, dim3 block, const A0& a0, const A1& a1, size_t lds_bytes)
{
    if (cx->profiling && cx->ev_used + 2 <= cx->ev.size()) {
        hipExtLaunchKernelGGL(kernel, grid, block, lds_bytes, cx->stream, cx->ev[cx->ev_used],
                              cx->ev[cx->ev_used + 1], 0, a0, a1);
        cx->ev_used += 2;
    } else {
        hipLaunchKernelGGL(kernel, grid, block, lds_bytes, cx->stream, a0, a1);
    }
}

template <typename Kern, typename Args>
void launch_main(Kern kernel, dim3 grid, dim3 block, const Args& args, size_t lds_bytes = 0)
{
    if (cx->profiling && cx->ev_used + 2 <= cx->ev.size()) {
        hipExtLaunchKernelGGL(kernel, grid, block, lds_bytes, cx->stream, cx->ev[cx->ev_used],
                              cx->ev[cx->ev_used + 1], 0, args);
        cx->ev_used += 2;
    } else {
        hipLaunchKernelGGL(kernel, grid, block, lds_bytes, cx->stream, args);
    }
}

// Every entry point that touches the device starts here: the device is made
// current for the calling thread and `cx` is the thread's context, created on
// the thread's first call.  ok() is false when that failed (out of memory) or
// the library is not initialised.  No lock is held afterwards: calls from
// different threads run side by side, each on its own stream.
struct Entered {
    bool good = false;
    Entered();
    ~Entered()
    {
        if (good) cx->depth.store(cx->depth.load(std::memory_order_relaxed) - 1, std::memory_order_relaxed);
    }
    Entered(const Entered&) = delete;
    Entered& operator=(const Entered&) = delete;
    bool ok() const { return good; }
};

#define ENTER()                                   \
    Entered entered_;                             \
    if (!entered_.ok()) return g.inited ? WR_HIP_ERR_NOMEM : WR_HIP_ERR_STATE


}  // namespace wr
