// fake_hip.hpp — controls and counters of fake_hip.cpp.
#pragma once

#include <atomic>
#include <cstddef>
#include <cstdint>
#include <vector>

namespace fake {
// bytes of device memory from here on, and the number of the hipMalloc call
// (counted from here) that fails whatever is left (0: none)
void reset(size_t capacity = ~(size_t)0, size_t fail_at = 0);
size_t in_use();     // bytes of device memory
size_t n_mallocs();  // since reset
size_t n_pins();     // hipHostMalloc since reset
extern bool tiny;                         // whole solves in one launch where the planner wants them
extern std::vector<uint32_t> tiny_iters;  // iterations of each such launch
// packs: launches that pack fibers; on_null: copies and counts on the null stream
extern std::atomic<size_t> copies, launches, packs, on_null;
}  // namespace fake
