// regression.hpp -- the per-voxel regression of cdm_get_gradient 'r', shared
// by the 3-D and 2-D loops.
#pragma once

#include "device.hpp"
#include "div_count.hpp"

namespace tiplhip {

// Window sums of Js (j), It (i), their squares and product.
struct Sums5 {
    uint32_t j, i, jj, ii, ji;
};

// linear_regression (numerical/statistics.hpp:694-713) of It on Js over a
// window of `count` voxels, FULL of them away from the borders, in FP64 and in
// the reference's order: returns the factor of the image gradient (0 where the
// voxel takes no part) and sets its cost term.
template <int FULL>
__device__ inline float regress(uint32_t js, uint32_t it, const Sums5& s, int count, float& cost)
{
    if (js == 0u || it == 0u) return 0.0f;
    double dn = double(FULL), inv = 1.0 / double(FULL);
    if (count != FULL) {
        dn = double(count);
        inv = 1.0 / dn;
    }
    const double mean_x = div_count(s.j, dn, inv);
    const double mean_y = div_count(s.i, dn, inv);
    const double x_var = div_count(s.jj, dn, inv) - mean_x * mean_x;
    const double y_var = div_count(s.ii, dn, inv) - mean_y * mean_y;
    if (x_var == 0.0 || y_var == 0.0) return 0.0f;
    const double cov = div_count(s.ji, dn, inv) - mean_x * mean_y;
    const float a = float(cov / x_var);
    if (!(a > 0.0f)) return 0.0f;
    const float b = float(mean_y - double(a) * mean_x);
    const float r2 = float(cov * cov / x_var / y_var);
    float sc = float(js) * a;
    sc = sc + b;
    sc = sc - float(it);
    sc = r2 * sc;
    cost = -r2;
    return sc;
}

}  // namespace tiplhip
