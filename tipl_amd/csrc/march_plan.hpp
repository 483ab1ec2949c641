// march_plan.hpp -- how the kernels that march z split a volume's planes.  Plain
// C++ (no HIP), so the plan is tested on a CPU-only host.
#pragma once

#include <algorithm>
#include <cstdint>

namespace tiplhip {

struct MarchPlan {
    uint32_t runs;  // z runs of every column
    int planes;     // planes of a run
    int tried;      // candidates looked at
};

// The number of z runs, of at least `least` planes each, with the fewest steps
// over all rounds of `resident` workgroups: every one of `cols` columns has its
// runs, and a run of p planes takes p + ramp steps.  Where a round holds several
// runs of every column, a number of rounds does best with the most it holds: one
// candidate for each number, else one for each number of runs, 64 in all (what
// more could save is the idle part of the last of 64 rounds).  A search over the
// lengths would look at a volume's depth of them, a launch.
inline MarchPlan march_plan(uint32_t cols, int d, int ramp, int least, uint32_t resident)
{
    least = std::min(least, d);
    MarchPlan m{1, d, 0};
    uint64_t best = ~uint64_t(0);
    for (uint64_t k = 1; k <= 64; ++k) {
        uint64_t runs = std::min<uint64_t>(cols < resident ? k * resident / cols : k, uint64_t(d));
        const int planes = std::max(least, int((uint64_t(d) + runs - 1) / runs));
        runs = (uint64_t(d) + uint64_t(planes) - 1) / uint64_t(planes);
        const uint64_t rounds = (cols * runs + resident - 1) / resident;
        const uint64_t steps = rounds * uint64_t(planes + ramp);
        ++m.tried;
        if (steps < best) {
            best = steps;
            m.runs = uint32_t(runs);
            m.planes = planes;
        }
        if (planes == least) break;
    }
    return m;
}

}  // namespace tiplhip
