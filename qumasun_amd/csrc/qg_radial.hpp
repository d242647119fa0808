// qg_radial.hpp — tabulated radial functions of the projectors, the same source for the host tables
// (qg_setup.cpp) and the device lists (qg_sphere.hip); also compiled by the tests without HIP.
#pragma once
#include <cmath>

#if defined(__HIPCC__) || defined(__HIP__)
#define QG_HD __host__ __device__
#else
#define QG_HD
#endif

namespace qg {

// RadialGrid2::GetValueByXi (RadialGrid2.h:81-136) at rel = xi - xi_min of n >= 5 values: linear in the
// outer intervals, cubic Hermite next to them, quintic Hermite with 4th-order derivative estimates
// inside, zero beyond the last point.  Below the first point (r_min may lie below exp(xi_min), or equal
// it but for rounding) the first value, as for r < r_min: no interval is read there.
QG_HD inline double radial_by_rel(double rel, const double* v, int n, double xi_delta) {
    const double fl = floor(rel / xi_delta);
    if (!(fl >= 0.0)) return v[0];
    if (fl >= (double)(n - 1)) return 0.0;
    const int i = (int)fl;
    if (i == 0 || i == n - 2) {
        const double t = rel / xi_delta - fl;
        return v[i] * (1.0 - t) + v[i + 1] * t;
    }
    const double t = rel / xi_delta - (double)i;
    if (1 < i && i < n - 3) {
        const double fm2 = v[i - 2], fm1 = v[i - 1], f0 = v[i], f1 = v[i + 1], f2 = v[i + 2], f3 = v[i + 3];
        const double g0 = 2.0 / 3.0 * (f1 - fm1) - 1.0 / 12.0 * (f2 - fm2);
        const double g1 = 2.0 / 3.0 * (f2 - f0) - 1.0 / 12.0 * (f3 - fm1);
        const double h0 = 4.0 / 3.0 * (f1 + fm1) - 1.0 / 12.0 * (f2 + fm2) - 5.0 / 2.0 * f0;
        const double h1 = 4.0 / 3.0 * (f2 + f0) - 1.0 / 12.0 * (f3 + fm1) - 5.0 / 2.0 * f1;
        const double e0 = f1 - (f0 + g0 + h0 / 2.0);
        const double e1 = g1 - (g0 + h0);
        const double e2 = h1 - h0;
        const double a3 = 10.0 * e0 - 4.0 * e1 + 0.5 * e2;
        const double a4 = -15.0 * e0 + 7.0 * e1 - e2;
        const double a5 = f1 - f0 - g0 - h0 / 2.0 - a3 - a4;
        return f0 + t * (g0 + t * (h0 / 2.0 + t * (a3 + t * (a4 + t * a5))));
    }
    const double v0 = v[i], v1 = v[i + 1];
    const double s1 = (v[i + 2] - v0) / 2.0, s0 = (v1 - v[i - 1]) / 2.0;
    const double a = s1 + s0 - 2.0 * (v1 - v0);
    const double b = -s1 - 2.0 * s0 + 3.0 * (v1 - v0);
    return a * t * t * t + b * t * t + s0 * t + v0;
}

}  // namespace qg
