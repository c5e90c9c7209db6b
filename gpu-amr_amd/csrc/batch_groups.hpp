// batch_groups.hpp -- how a batch's trees are split into groups (host code).
#pragma once

#include <cstddef>
#include <cstdint>
#include <vector>

namespace amrhip
{

// First item of every run when consecutive items of the given sizes are packed
// into runs of at most `most`, each filled until the next item would not fit.
// An item larger than that is a run of its own.
inline std::vector<size_t> fill_runs(std::vector<uint64_t> const& size, uint64_t most)
{
    std::vector<size_t> first;
    uint64_t            fill = 0;
    for (size_t i = 0; i < size.size(); ++i)
    {
        if (first.empty() || size[i] > most || fill > most - size[i])
        {
            first.push_back(i);
            fill = 0;
        }
        fill += size[i];
    }
    return first;
}

// The same with no more runs than that, but the largest run as small as it can
// be: filling up leaves a last run of any size.
inline std::vector<size_t> even_runs(std::vector<uint64_t> const& size, uint64_t most)
{
    const size_t fewest = fill_runs(size, most).size();
    uint64_t     lo = 0, hi = most; // the least limit that needs no more runs
    while (lo < hi)
    {
        const uint64_t mid = lo + (hi - lo) / 2;
        if (fill_runs(size, mid).size() <= fewest)
            hi = mid;
        else
            lo = mid + 1;
    }
    return fill_runs(size, hi);
}

} // namespace amrhip
