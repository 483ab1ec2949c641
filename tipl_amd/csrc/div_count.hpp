// div_count.hpp -- exact division of a window sum by the window's size.
#pragma once

#include <cstdint>

namespace tiplhip {

#if defined(__HIPCC__)
#define TIPLHIP_HOST_DEVICE __host__ __device__
#else
#define TIPLHIP_HOST_DEVICE
#endif

// s / dn correctly rounded, from inv = 1 / dn rounded: one Newton step on the
// quotient with an exact remainder (Markstein's theorem), three operations
// where the general FP64 division takes about eleven.  Compared with the
// division for every window size and every sum in tests/test_div_count.py.
TIPLHIP_HOST_DEVICE inline double div_count(uint32_t s, double dn, double inv)
{
    const double a = double(s);
    const double q = a * inv;
    return __builtin_fma(__builtin_fma(-q, dn, a), inv, q);
}

}  // namespace tiplhip
