// SPDX-License-Identifier: MIT
//
// Size limits of the persistent launches, shared by the host library and the
// CPU tests (plain C++, no HIP headers).
//
#pragma once

#include <cstdint>

namespace cgs
{

// Persistent kernels run 256-thread workgroups (4 waves of 64).  Each wave
// takes `perFetch` work items at a time from a 32-bit counter with one
// atomicAdd, and stops at the first fetch past the end: the counter ends at
// most at items + waves × perFetch.  A launch is refused unless that stays
// below 2^32, so the counter never wraps and restarts a wave at item 0.
inline bool counterFits(uint64_t items, uint64_t grid, uint64_t perFetch)
{
    const uint64_t waves = grid * 4;
    return items < (1ull << 32) && perFetch < (1ull << 32) && waves < (1ull << 32) &&
           items + waves * perFetch < (1ull << 32);
}

// Whether a sub-patch call of n patches has each lane move its own patch
// (kSubpatchFew) rather than a wave move its 64 through LDS (kSubpatch): up to
// two waves per CU of 256, whose patches (16 KiB a wave) its 32-KiB L1 holds.
// Per lane against through LDS: 100 patches 4.3 and 6.4 us, 10,000 5.1 and 7.0,
// 20,000 6.5 and 7.4, 50,000 10.4 and 8.6, 300,000 37.5 and 31.0.
inline bool subpatchPerLane(uint32_t n) { return n <= 2 * 256 * 64; }

// Work items of a render: one per pixel of every 8×8 tile (edge tiles whole).
inline uint64_t renderItems(uint32_t w, uint32_t h)
{
    return (((uint64_t)w + 7) / 8) * (((uint64_t)h + 7) / 8) * 64;
}

} // namespace cgs
