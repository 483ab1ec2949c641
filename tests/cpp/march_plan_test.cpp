// march_plan against a search over every length of run: the same number of
// steps for volumes of up to 512 planes, at most 1 / 64 more for any, and few
// candidates whatever the depth.
#include "../../tipl_amd/csrc/march_plan.hpp"

#include <cstdio>
#include <cstdlib>

namespace {

uint64_t steps_of(uint32_t cols, int d, int planes, int ramp, uint32_t resident)
{
    const uint64_t runs = uint64_t(d + planes - 1) / uint64_t(planes);
    return (cols * runs + resident - 1) / resident * uint64_t(planes + ramp);
}

bool check(uint32_t cols, int d, int ramp, int least, uint32_t resident)
{
    const tiplhip::MarchPlan m = tiplhip::march_plan(cols, d, ramp, least, resident);
    uint64_t best = ~uint64_t(0);
    for (int planes = d; planes >= std::min(least, d); --planes)
        best = std::min(best, steps_of(cols, d, planes, ramp, resident));
    const bool covers = m.planes >= 1 && uint64_t(m.runs) * uint64_t(m.planes) >= uint64_t(d) &&
                        uint64_t(m.runs - 1) * uint64_t(m.planes) < uint64_t(d);
    const uint64_t got = steps_of(cols, d, m.planes, ramp, resident);
    if (covers && (got == best || (d > 512 && got * 64 <= best * 65))) return true;
    std::printf("cols %u d %d ramp %d least %d: %u runs of %d\n", cols, d, ramp, least, m.runs, m.planes);
    return false;
}

}  // namespace

int main()
{
    for (int d = 1; d <= 512; ++d)
        for (uint32_t cols : {1u, 2u, 3u, 12u, 45u, 120u, 511u, 512u, 513u, 2400u, 30000u})
            if (!check(cols, d, 10, 2, 512) || !check(cols, d, 14, 1, 512)) return 1;
    srand(1);
    for (int i = 0; i < 3000; ++i)
        if (!check(1u + uint32_t(rand()) % 4000u, 1 + rand() % 3000, 1 + rand() % 20, 1 + rand() % 4,
                   1u + uint32_t(rand()) % 1000u))
            return 1;
    // one call a launch: a deep volume must not take longer to plan than to run
    for (int d : {1, 1000, 100000, 1 << 20, 178956000})
        for (uint32_t cols : {3u, 511u, 512u, 100000u})
            if (tiplhip::march_plan(cols, d, 10, 2, 512).tried > 64) return 1;
    std::printf("march plan ok\n");
    return 0;
}
