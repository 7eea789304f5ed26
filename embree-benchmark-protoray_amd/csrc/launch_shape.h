// launch_shape.h -- workgroups of a launch that is traced in groups of 8 lanes
// from its start, and whether they need work counters.  Plain host arithmetic.
#pragma once

#include <stdint.h>

#include <algorithm>

namespace prt {

// Launches of at most this many items are traced in groups of 8 lanes from
// their start: with so few, a launch takes as long as its longest path's chain
// of steps, and a step of a group is shorter.  Above, throughput decides: a
// group's 8 lanes do the work of one.  Measured lane by lane / in groups, us:
//   closest hits  512 rays 112 / 73, 8192 144 / 92, 32768 172 / 104,
//                 49152 174 / 177, 65536 173 / 217
//   primary       9216 74 / 46, 32256 83 / 82, 64000 107 / 126
//   diffuse       32256 265 / 172, 64000 324 / 279, 96000 584 / 473, 286 /
//                 283, 324 / 319 (three scenes), 140000 314 / 356
//   diffuse2      32256 425 / 317, 64000 467 / 381, 96000 939 / 762, 454 /
//                 409, 140000 484 / 494
// The albedo modes trace the same paths as diffuse.
constexpr uint64_t kSpreadRays = 32768, kSpreadPaths = 96 << 10;
constexpr uint64_t kSpreadRun = 8;  // items that a wave takes at once: one per group

// Workgroups of such a launch: a wave per 8 items, on as many CUs as there are
// waves, then up to all waves of each, `most` workgroups in all.
inline int spread_grid(int num_cus, uint64_t items, int block_waves, int most)
{
    const int waves = (int)std::min<uint64_t>((items + kSpreadRun - 1) / kSpreadRun, 1u << 30);
    return std::min(most, std::max(1, std::max(std::min(waves, num_cus), (waves + block_waves - 1) / block_waves)));
}

// Every item belongs to the first run of some wave, so that the launch reads no
// work counter.  32768 items are the 4096 runs of 256 CUs with 4 workgroups of 4
// waves each; with fewer CUs or workgroups a smaller launch is the most that is
// covered.
inline bool spread_covers(int grid, int block_waves, uint64_t items)
{
    return (uint64_t)std::max(grid, 0) * (uint64_t)block_waves >= (items + kSpreadRun - 1) / kSpreadRun;
}

}  // namespace prt
