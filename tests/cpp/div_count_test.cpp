// div_count against the division, for every size of a border-clipped 5x5x5
// window and every sum such a window can hold (at most 255 * 255 a voxel).
#include "../../tipl_amd/csrc/div_count.hpp"

#include <cstdio>
#include <set>

int main()
{
    std::set<int> counts;
    for (int x = 1; x <= 5; ++x)
        for (int y = 1; y <= 5; ++y)
            for (int z = 1; z <= 5; ++z) counts.insert(x * y * z);
    unsigned long long checked = 0;
    for (int c : counts) {
        const double dn = double(c), inv = 1.0 / dn;
        for (uint32_t s = 0; s <= uint32_t(c) * 65025u; ++s, ++checked)
            if (tiplhip::div_count(s, dn, inv) != double(s) / dn) {
                std::printf("count %d sum %u differs\n", c, s);
                return 1;
            }
    }
    std::printf("div_count ok (%llu quotients)\n", checked);
    return 0;
}
