// Follows the ray indices of traversal launches on the host (ray_grid.h): for n
// rays, launched in parts of at most kMaxLaunch, `wave_rays` of them per
// wavefront and a grid limit, prints
//   parts-with-too-many-threads  wrong-places  wrong-rays  most-rays-a-lane
// The loop is the kernels': 32-bit, from a lane's first ray in steps of the
// whole grid's.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../povray_amd/csrc/ray_grid.h"

using namespace pvx;

int main(int argc, char **argv) {
    const uint64_t all = std::strtoull(argv[1], nullptr, 10);
    const uint32_t r = (uint32_t)std::atoi(argv[2]), limit = (uint32_t)std::strtoull(argv[3], nullptr, 10);
    uint64_t threads_bad = 0, wrong_places = 0, wrong_rays = 0, most = 0, covered = 0;
    for (uint64_t at = 0; at < all; at += kMaxLaunch) {
        const uint32_t n = (uint32_t)std::min<uint64_t>(all - at, kMaxLaunch);
        covered += n;
        const uint32_t units = launch_units(n, r, limit), blocks = units * (kBlock / kWaveBlock);
        threads_bad += units == 0 || (uint64_t)units * kBlock > 0xFFFFFFFFull;
        // every place is some block's: the lanes' first rays are 0 .. blocks * r - 1
        std::vector<bool> taken(blocks, false);
        for (uint32_t b = 0; b < blocks; b++) {
            const uint32_t p = xcd_place(b, blocks);
            if (p >= blocks || taken[p])
                wrong_places++;
            else
                taken[p] = true;
        }
        // a lane's rays: i0, i0 + step, ... below n, each once (the lanes of the
        // first, the last and some blocks in between)
        const uint32_t step = blocks * r;
        const uint64_t wide = (uint64_t)blocks * r;
        for (uint32_t b = 0; b < blocks; b += b < 300 || b + 300 > blocks ? 1 : std::max(1u, (blocks - 600) / 200)) {
            for (uint32_t lane = 0; lane < r; lane += r > 1 ? r - 1 : 1) {
                const uint64_t i0 = (uint64_t)xcd_place(b, blocks) * r + lane;
                uint64_t want = i0, seen = 0;
                for (uint32_t i = (uint32_t)i0; i < n && seen < (1u << 20); i += step, want += wide, seen++)
                    wrong_rays += want >= n || i != want;
                wrong_rays += want < n; // ended early
                most = std::max(most, seen);
            }
        }
    }
    wrong_rays += covered != all;
    std::printf("%llu %llu %llu %llu\n", (unsigned long long)threads_bad, (unsigned long long)wrong_places,
                (unsigned long long)wrong_rays, (unsigned long long)most);
    return 0;
}
