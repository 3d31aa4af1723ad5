// Who takes a decode step's layers in one launch, and when (wr_hip_attn_step_dev): host code only.
#pragma once

#include <atomic>
#include <cstdint>

namespace wr {

// One off a counter that several threads count down: false, and nothing taken, when it is at zero.
inline bool count_down(std::atomic<uint32_t>& n)
{
    uint32_t v = n.load(std::memory_order_relaxed);
    while (v && !n.compare_exchange_weak(v, v - 1, std::memory_order_relaxed)) {
    }
    return v != 0;
}

}  // namespace wr
