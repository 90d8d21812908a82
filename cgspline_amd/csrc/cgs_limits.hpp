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

// Work items that a wave of a persistent launch of at most `grid` workgroups
// takes at a time: 64, one per lane, and fewer (down to 8, a power of two) where
// that still gives every wave some.  A wave waits for its slowest item, and its
// lanes without one share the others' clips: a 64-ray pick took 71 us this way
// and 91 us in one wave, 5,000 shaded rays 640 and 1,408 us, a 200x150 frame of
// 19 lights 3.7 and 10.3 ms, a 256x256 one-light frame 305 and 336 us.
inline uint32_t launchChunk(uint64_t items, uint32_t grid)
{
    uint32_t chunk = 64;
    while (chunk > 8 && items <= (uint64_t)grid * 4 * (chunk / 2)) chunk /= 2;
    return chunk;
}

// Workgroups of a persistent launch of `items` work items, `chunk` at a time to
// a wave: as many as have some, at most `grid`.  A wave without work still adds
// to the launch's one counter, which takes about 10 ns each: a 64-ray pick took
// 85 us of 768 workgroups, 74 us of 512, 70 us of the 2 that have rays.
inline uint32_t launchGrid(uint64_t items, uint32_t grid, uint32_t chunk)
{
    const uint64_t need = (items + 4ull * chunk - 1) / (4ull * chunk);
    return need >= grid ? grid : need ? (uint32_t)need : 1u;
}

// Whether a batched launch of `rays` rays takes the kernels of two waves per SIMD
// rather than three: up to ten rays for each lane of two waves on the 256 CUs.
// Then most waves hold the launch's camera rays, whose clips the spills of three
// waves slow down; above, the scattered rays' walks need the third.  Two against
// three: 150,000 rays 249 and 267 us, 660,000 387 and 424, 1.0M 434-491 and
// 447-514, 1.9M 807-998 and 772-932, 3.4M 1,070 and 1,025, 17M 7.1 and 6.3 ms.
inline bool batchAtTwoWaves(uint64_t rays) { return rays <= 10ull * 256 * 512; }

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
