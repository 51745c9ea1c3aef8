// Which rays a wavefront of the traversal kernels takes, and how many blocks a
// launch has.  Ray counts go up to 2^32 - 1, and neither the kernels' ray index
// nor a launch's threads may leave 32 bits.  Plain arithmetic that also builds
// for the host.
#ifndef PVX_RAY_GRID_H
#define PVX_RAY_GRID_H

#include <cstddef>
#include <cstdint>

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define PVX_GRID_FN __host__ __device__ __forceinline__
#else
#define PVX_GRID_FN inline
#endif

namespace pvx {

constexpr int kBlock = 256;      // lanes per unit of a traversal grid (threads per block of the kd walk)
// Threads per block of the BVH walks: one wavefront, so that its place is
// free for the next one as soon as it ends (a kBlock unit is four of them).
constexpr int kWaveBlock = 64;

// A walk whose stack cannot outgrow its LDS entries needs no spill area per
// resident lane, so its launch covers all rays (kWholeGrid) instead of a
// persistent grid: the hardware then hands out wavefronts as others end.  A
// persistent grid with a fixed stride left less than half of its places
// filled (camera rays of the 1.3M-triangle icosphere: 2.3 of 5 wavefronts per
// SIMD on average).  2^22 units are 2^30 threads.
constexpr uint32_t kWholeGrid = 1u << 22;

// Rays of one launch at most: larger counts are launched in parts.  A lane goes
// from ray i to ray i + (rays of the whole grid) <= 2^31 + 2^30, which 32 bits
// hold.  (Asking instead, per ray, whether another whole step is left cost the
// camera rays of the 1.3M-triangle icosphere 1.4 %.)
constexpr uint32_t kMaxLaunch = 1u << 31;

// Blocks go to the eight XCDs in turn, each with an L2 of its own: the place
// of block b's rays such that sixteen neighbouring wavefronts (of rays
// that mostly walk the same nodes) share one (camera rays of the
// 1.3M-triangle icosphere 568 -> 556 us, its reflections at 327,680 triangles
// 253 -> 242 us; 4 or 64 neighbours: 571 and 560, 245 and 241 us).  Blocks past
// the last whole group keep their place.
PVX_GRID_FN uint32_t xcd_place(uint32_t b, uint32_t grid) {
    constexpr uint32_t kXcds = 8, kRun = 16;
    const uint32_t whole = grid / (kXcds * kRun) * (kXcds * kRun);
    return b < whole ? (b / (kXcds * kRun) * kXcds + b % kXcds) * kRun + b / kXcds % kRun : b;
}

// Rays per wavefront of a launch of n rays on a grid of `grid` units: 64,
// halved while the grid still holds every wavefront at once.  A wavefront
// runs every path that any of its rays takes, so below a full grid fewer rays
// each end sooner (plain radiosity of the 5,000-box room, whose rounds gather
// some ten thousand rays: 53 ms with 64 rays per wavefront, 45 ms so).
inline uint32_t rays_per_wave(size_t n, uint32_t grid) {
    uint32_t r = 64;
    while (r > 1 && n <= (size_t)grid * (kBlock / kWaveBlock) * (r / 2)) r /= 2;
    return r;
}

// Units of a launch of n rays with `wave_rays` of them per wavefront, at most
// `grid`.
inline uint32_t launch_units(size_t n, uint32_t wave_rays, uint32_t grid) {
    const size_t per = (size_t)(kBlock / kWaveBlock) * wave_rays, units = (n + per - 1) / per;
    return units < grid ? (uint32_t)units : grid;
}

} // namespace pvx

#endif
