// gg_sizing.hpp -- sizes and offsets of a call's buffers (host arithmetic
// only, no device code: a plain C++ compiler builds it).
#pragma once

#include <algorithm>
#include <cstddef>
#include <vector>

namespace gg {

// The autotuner's trial grids, one allocation: job j's grid of
// sizes[j] x sizes[j] cells starts at cell offsets[j].  Returns the cells of
// all of them.  (In size_t throughout: 129 grids of 4096^2, 33 of 8192^2 or 9
// of 16384^2 pass 2^31 cells.)
inline size_t place_grids(const std::vector<int>& sizes, std::vector<size_t>& offsets)
{
    size_t cells = 0;
    offsets.clear();
    for (const int g : sizes)
    {
        offsets.push_back(cells);
        cells += (size_t)g * (size_t)g;
    }
    return cells;
}

// Partial regions (slots) that c visits over `tiles` tiles can need, in items
// of V visits: a tile of c_t visits has ceil(c_t / V) items, and slots only
// when that is 2 or more; such tiles hold more than V visits each, so that
// there are at most c / V of them, and each adds less than one to c_t / V.
inline unsigned long long slot_bound(unsigned long long c, unsigned long long tiles,
        unsigned long long V)
{
    return c / V + std::min(tiles, c / V);
}

// Band kernel: visits per work item.  An item is worked on by 32 waves, one
// per band of 8 rows and column block, so a small call needs small items to
// fill the chip (kernel and merge, 2,003 visibilities: 157 us with items of
// 1024 visits, 38 us with 64; 200,000: 269 us with 1024, 221 us with 512),
// a large one fewer partial regions to merge (13.2M in 24 grids: 23.7 ms with
// 512, 23.0 ms with 1024, 23.9 ms with 2048).  Up to 65,536 visibilities the
// size keeps the partial regions below about 200 (50 MiB).
inline unsigned band_visits_per_item(unsigned long long num_points)
{
    if (num_points > 65536)
        return num_points < 524288 ? 512u : num_points < (16ull << 20) ? 1024u : 4096u;
    unsigned v = 64;
    while (v * 128ull < num_points) v <<= 1;
    return v;
}

struct JobSize
{
    unsigned long long points, tiles;
};

// The band kernel's item size of each job of a call.  Up to kOwnItemJobs jobs
// take the size that a call of their own would.  More jobs than that fill the
// chip together, and small items only add partial regions to write and merge:
// they take at least the size of one call of all their visibilities, up to
// 1024 (pass of 1000 jobs of 8192 visibilities on 1024^2: 31.6 ms with their
// own size of 64, 12.7 with 1024; 1500 of 2000 on 512^2: 16.3 and 7.3; 64 of
// 600,000 on 4096^2: 73.8 with 1024, 77.4 with 2048, 83.1 with 4096).
// Beyond that all sizes rise until the partial regions that a captured pass
// has to allow for (per_point: the tiles one footprint can touch) are within
// kSlotBudget, but not beyond `coarsest`, the size the other kernels would
// take.  The budget, a sixth of the device's memory, is what the 64 jobs above
// need for their fastest size (44.6 GiB captured; an eager pass, that knows the
// counts, allocates a third).  All from the call's shape alone, so that
// captured, eager and repeated passes split the work alike.
constexpr size_t kOwnItemJobs = 8;
constexpr unsigned long long kSlotBudget = 48ull << 30;

inline void band_item_sizes(const std::vector<JobSize>& jobs, unsigned long long per_point,
        unsigned long long slot_bytes, unsigned coarsest, std::vector<unsigned>& sizes)
{
    unsigned long long all = 0;
    for (const JobSize& j : jobs) all += j.points;
    unsigned least = jobs.size() > kOwnItemJobs ? std::min(band_visits_per_item(all), 1024u) : 64u;
    sizes.resize(jobs.size());
    for (;; least *= 2)
    {
        unsigned long long slots = 0;
        for (size_t i = 0; i < jobs.size(); ++i)
        {
            sizes[i] = std::max(band_visits_per_item(jobs[i].points), least);
            slots += slot_bound(jobs[i].points * per_point, jobs[i].tiles, sizes[i]);
        }
        if (slots <= kSlotBudget / slot_bytes || least >= coarsest) return;
    }
}

} // namespace gg
