// Entries of the flow tracing's border tables and the hop from one to the
// next.  Plain constexpr code: the device's, and a host program's.
#pragma once

#include <cstdint>

namespace cageo {

constexpr uint32_t K_LOCAL = 0, K_RESOLVED = 1, K_EXIT = 2, K_STUCK = 3;
constexpr uint64_t STEP_MASK = (1ull << 30) - 1;

constexpr uint64_t pack(uint32_t kind, uint32_t steps, int32_t value) {
    return ((uint64_t)kind << 62) | ((uint64_t)(steps & STEP_MASK) << 32) |
           (uint64_t)(uint32_t)value;
}
constexpr uint32_t kind_of(uint64_t e) { return (uint32_t)(e >> 62); }
constexpr uint32_t steps_of(uint64_t e) { return (uint32_t)((e >> 32) & STEP_MASK); }
constexpr int32_t value_of(uint64_t e) { return (int32_t)(uint32_t)e; }

// Follow entry e one hop through entry f (the entry of e's target).  The
// steps saturate.
constexpr uint64_t hop(uint64_t e, uint64_t f) {
    const uint32_t k = kind_of(f), s = steps_of(e) + steps_of(f);
    if (k == K_STUCK) return pack(K_STUCK, 0, 0);
    return pack(k, s > STEP_MASK ? (uint32_t)STEP_MASK : s, value_of(f));
}

// Whether a chain that is still at an exit after `steps` steps is taken for a
// cycle: more steps than its raster has cells, or more than an entry holds
// (on a raster of 2^30 - 1 cells or more no chain would reach the former).
constexpr bool is_cycle(uint32_t steps, uint32_t cells) {
    return steps > (cells < STEP_MASK ? cells : (uint32_t)STEP_MASK - 1u);
}

}  // namespace cageo
