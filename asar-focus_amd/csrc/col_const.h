// FP64 constants of one range column (ColConst) and the bound on the RCMC shift over all columns.
#pragma once

#include <climits>

#include "kernels.h"
#include "poly.h"

namespace asarf {

// Column x's constants from the Doppler polynomial dc3 (highest power first) into a.col, and the wave's largest shift
// bound into *a.reach. Every lane of the wave calls it (lanes past the last column take part in the reduction).
__device__ __forceinline__ void col_const_store(const ColConstArgs& a, int x, const double* dc3) {
    const bool valid = x < a.nrv;
    int r = 0;
    if (valid) {
        const double step = a.prf / (double)a.nbins;
        const double dc = polyval(dc3, 3, (double)x);
        const double r0 = a.r_first + (double)x * a.range_spacing;
        const double vr = polyval(a.vr_poly, 3, (double)x);
        ColConst c;
        c.dc = dc;
        c.dc_off = round(dc / step) * step;
        c.shift_k = a.wavelength * a.wavelength * r0 / (8.0 * vr * vr * a.range_spacing);
        c.inv_ka = a.wavelength * r0 / (2.0 * vr * vr);
        c.shift_b2 = c.shift_k * step * step;
        // Undefined statistics (a constant channel) leave no centroid: the fused core, which tests the band on whole
        // bins, then gets a band about 0 and a phase that is NaN, so that the column is NaN as with the FP64 band test
        // of the separate kernels, and not zero.
        const bool known = dc - dc == 0.0;
        c.turns_b2 = known ? 0.5 * c.inv_ka * step * step : dc - dc;
        c.m_dc = known ? (int)fmin(fmax(round(dc / step), -1e9), 1e9) : 0;
        // alias_about_dc's comparisons of kb * step with the band limits, as whole bins
        const double half = 0.5 * a.prf;
        c.alias_hi = INT_MAX;
        c.alias_lo = INT_MIN;
        if (dc < 0.0) {
            const double lim = half + dc;
            double k = floor(fmin(fmax(lim / step, -1e9), 1e9));
            if ((k + 1.0) * step <= lim) k += 1.0;
            if (k * step > lim) k -= 1.0;
            c.alias_hi = (int)k;
        } else if (dc > 0.0) {
            const double lim = -half + dc;
            double k = ceil(fmin(fmax(lim / step, -1e9), 1e9));
            if ((k - 1.0) * step >= lim) k -= 1.0;
            if (k * step < lim) k += 1.0;
            c.alias_lo = (int)k;
        }
        c.pad = 0;
        a.col[x] = c;
        // The aliased bin frequency stays within prf/2 of the centroid, so |f| <= prf/2 + |dc| bounds the
        // shift of every bin (plus one pixel against rounding).
        const double fmax = (0.5 * a.prf + fabs(dc)) * (1.0 + 1e-12);
        const double smax = c.shift_k * fmax * fmax;
        r = (smax >= 0.0 && smax < 1e6) ? (int)floor(smax + 0.5) + 1 : 1000000;
    }
    if (a.reach) {
        // one atomic per wave; every lane of the wave takes part in the reduction
        for (int o = 32; o > 0; o >>= 1) r = max(r, __shfl_xor(r, o));
        if ((threadIdx.x & 63) == 0 && r > 0) atomicMax(a.reach, r);
    }
}

}  // namespace asarf
