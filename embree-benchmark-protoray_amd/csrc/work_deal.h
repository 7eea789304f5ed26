// work_deal.h -- which work items belong to which counter of a persistent
// launch.  Items are dealt in runs of 2^run_lg; every 16 runs go to the 16
// counters, one each, in an order that shifts from one 16 to the next.
//
// The shift is what keeps the counters even.  A run of a frame is one 8x8 tile
// in row order.  With run r at counter r mod 16 a counter owned whole columns of
// tiles wherever a row has a multiple of 16 of them, in every sample of a job,
// and since the waves of a large launch stop with their own counter, the launch
// lasted as long as the heaviest columns.  The shift of the k-th 16 is the top of
// k times the fraction of sqrt(2): multiples of an irrational that no small
// fraction comes near spread evenly, whatever the rows' length.  Heaviest counter over
// the mean, frames of 4 to 512 tiles by 64 with columns of unequal cost, worst /
// average: no shift 3.69 / 1.53, sum of k's hexadecimal digits 1.64 / 1.09, this
// 1.23 / 1.05.  Job sets, us, while one counter served them all / no shift /
// this: 32 of 128x128 at 16 samples 3466 / 3646 / 3042, looking past most of the
// scene 3057 / 3859 / 2144, 16 of 256x256 5656 / 5232 / 4439.  What it costs: a
// workgroup's counters no longer keep to columns of tiles, so an XCD's L2 sees more
// of a scene.  32 scenes of 10.6 M triangles in one launch miss it 1458 M times
// instead of 942 M, 58.5 -> 58.9 ms (in workgroups of 128 59.8 -> 59.3); frames of
// 1.3 M triangles miss as often as before.
#pragma once

#include <stdint.h>

#include "prt_math.h"

namespace prt {

// Work counters of a persistent launch: 16 of them, a 128 B line each.
constexpr uint32_t kWorkCountersLg = 4;
constexpr uint32_t kWorkCounterStride = 32;
constexpr int kWorkWords = (int)kWorkCounterStride << kWorkCountersLg;
constexpr uint32_t kWorkCounterLast = (1u << kWorkCountersLg) - 1u;

PRT_HD uint32_t deal_shift(uint32_t k) { return (k * 0x6a09e667u) >> (32 - kWorkCountersLg); }

// The counter of run r, which is its (r / 16)-th run.
PRT_HD uint32_t deal_counter(uint32_t r)
{
    return (r - deal_shift(r >> kWorkCountersLg)) & kWorkCounterLast;
}

// The k-th run of counter c.
PRT_HD uint32_t deal_run(uint32_t c, uint32_t k)
{
    return (k << kWorkCountersLg) | ((c + deal_shift(k)) & kWorkCounterLast);
}

// How many of the first `runs` runs are counter c's.
PRT_HD uint32_t dealt_runs(uint32_t c, uint32_t runs)
{
    const uint32_t k = runs >> kWorkCountersLg;
    return k + ((deal_run(c, k) < runs) ? 1u : 0u);
}

}  // namespace prt
