// spectral_math.hpp -- the reciprocal-space multipliers, evaluated in FP64 for
// every storage precision, as the line passes apply them between a forward and
// an inverse transform (line_pass.hpp): the parts that a line shares first, the
// sines from a table.  The standalone multiplier kernel (spectral.hip) shares
// signed_wavenumber only and evaluates its element's multiplier whole, sines by
// sinpi; the two are compared for every kind in test_gpu_spectral_solve.py
// (test_solve_is_the_three_calls).
#pragma once

#include "common.hpp"
#include "kernels.hpp"

namespace zm {

__device__ __forceinline__ int signed_wavenumber(int k, int n) { return k <= n / 2 ? k : k - n; }

// The part of a multiplier that one line of the last transform axis shares:
// the sum of squared wavenumbers and of squared half-angle sines of the other
// axes, and the imaginary part of the dx4 symbol (2D, axis 0).
struct LineSymbol {
    double k2, h2, im;
};

// Kinds: 0 Poisson -1/|k|^2 (k = 0 -> 0), 1 heat exp(-p0 |k|^2 p1), 2 constant
// p0, 3 stencil symbol (Laplacian scale p0, dx4 delta p1), 4 Poisson times the
// stencil symbol.  A family is the code for several kinds: the kernels branch
// on it outside their loops, so that only the heat loop holds exp's constants.
//
// The stencil symbol is that of the periodic 5-/7-point Laplacian (scaled by
// p0) plus, in 2D, the 4th-order x-derivative [1, -8, 0, 8, -1] / (12 delta)
// when delta != 0: for the mode exp(2 pi i k x / N), theta = 2 pi k / N,
//   Laplacian: p0 * sum_d (2 cos theta_d - 2) = -4 p0 sum_d sin^2(theta_d / 2)
//   dx4:       i (8 sin theta_x - sin 2 theta_x) / (6 delta)
// (the sin^2 form has no cancellation at small k).  Axis 0 is the
// packed-column (gc) wavenumber, the axis zm_dx4 differentiates.
enum SpectralFamily { SF_PLAIN = 0, SF_HEAT = 1, SF_STENCIL = 2 };

// sin(pi q / n) from half_sin[f] = sin(pi s / n), s the signed wavenumber of f
__device__ __forceinline__ double sin_pi_over(const double* half_sin, int q, int n) {
    const int f = q & (n - 1), turns = q - signed_wavenumber(f, n);  // 0 mod n
    return turns & n ? -half_sin[f] : half_sin[f];
}

template <int FAMILY, bool ONLY_2D>
__device__ __forceinline__ LineSymbol line_symbol(const SpectralArgs& sp, int f0, int f1, int n) {
    LineSymbol ls{0.0, 0.0, 0.0};
    const bool d3 = !ONLY_2D && sp.dims == 3;
    const int s0 = signed_wavenumber(f0, n), s1 = signed_wavenumber(f1, n);
    ls.k2 = (double)s0 * s0 + (d3 ? (double)s1 * s1 : 0.0);
    if constexpr (FAMILY == SF_STENCIL) {
        double h = sp.half_sin[f0];
        ls.h2 = h * h;
        if (d3) {
            h = sp.half_sin[f1];
            ls.h2 += h * h;
        }
        if (sp.p1 != 0.0) {
            const double s1x = sin_pi_over(sp.half_sin, 2 * s0, n), s2x = sin_pi_over(sp.half_sin, 4 * s0, n);
            ls.im = (8.0 * s1x - s2x) / (6.0 * sp.p1);
            if (sp.conj) ls.im = -ls.im;
        }
    }
    return ls;
}

// The multiplier at frequency f of the last axis, h = half_sin[f] = sin(pi s /
// N) of its signed wavenumber s (read by the stencil family only).
template <int FAMILY>
__device__ __forceinline__ void line_multiplier(const SpectralArgs& sp, const LineSymbol& ls, int f, int n, double h,
                                                double* mr, double* mi) {
    const int s = signed_wavenumber(f, n);
    const double k2 = sp.kscale * sp.kscale * (ls.k2 + (double)s * s);
    *mi = 0.0;
    if constexpr (FAMILY == SF_HEAT) {
        *mr = exp(-sp.p0 * k2 * sp.p1);  // heat: exp(-nu |k|^2 dt)
    } else {
        const double poisson = (k2 == 0.0) ? 0.0 : -1.0 / k2;  // 1 / (-|k|^2), mean mode removed
        if constexpr (FAMILY == SF_PLAIN) {
            *mr = sp.kind == 0 ? poisson : sp.p0;
        } else {
            *mr = -4.0 * sp.p0 * (ls.h2 + h * h);
            *mi = ls.im;
            if (sp.kind == 4) {
                *mr *= poisson;
                *mi *= poisson;
            }
        }
    }
}

}  // namespace zm
