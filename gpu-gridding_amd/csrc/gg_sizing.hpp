// gg_sizing.hpp -- sizes and offsets of a call's buffers (host arithmetic
// only, no device code: a plain C++ compiler builds it).
#pragma once

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

} // namespace gg
