// The limits of the kernels with 32-bit byte offsets, against the offsets
// themselves in 64 bits: everything such a kernel forms stays as it is when
// cut to 32 bits up to the limit, and the first volume past it is refused
// before anything wraps.
#include "../../tipl_amd/csrc/field_limits.hpp"

#include <cstdint>
#include <cstdio>

using namespace tiplhip;

int main()
{
    const uint64_t last = ((uint64_t(1) << 32) - 1) / 12;  // 357913941
    for (uint64_t n = last - 3; n <= last + 3; ++n) {
        // the length of the buffer and the end of its last voxel
        const bool wraps = uint64_t(uint32_t(n) * 12u) != n * 12;
        if (field_fits_32(n) == wraps) {
            std::printf("%llu voxels\n", static_cast<unsigned long long>(n));
            return 1;
        }
    }
    if (field_fits_32(715ull * 708 * 708) || !field_fits_32(700ull * 700 * 700)) return 1;
    // marched tiles: six planes past the volume's first voxel of the last plane
    // (four sweeps, two planes of loads ahead), 27 rows and 58 columns past the
    // last row and column (a tile's first lies at most four before them)
    const int64_t shapes[][3] = {{1, 1, 178956000}, {560, 560, 560}, {563, 560, 560}, {1, 2700000, 64},
                                 {2, 1, 60000000},  {1000, 421, 421}, {16, 3000, 3500}, {1, 1, 2400000},
                                 {178956800, 1, 1}, {178956890, 1, 1}};
    for (const auto& s : shapes) {
        const int64_t w = s[2], wh = s[1] * s[2], n = s[0] * wh;
        if (!marched_field_fits(size_t(n), size_t(wh), size_t(w))) continue;
        const int64_t top = n - 1 + 6 * wh + 27 * w + 58;
        if (top * 12 >= (int64_t(1) << 31)) {
            std::printf("%lld x %lld x %lld\n", static_cast<long long>(s[2]), static_cast<long long>(s[1]),
                        static_cast<long long>(s[0]));
            return 1;
        }
    }
    std::printf("field limits ok\n");
    return 0;
}
