// Quotients of the exact gravity terms without branches, for operands in a
// window, bit for bit those of `sqrt` and `/`.
//
// A term is G m d / D^3 per component with D = sqrt(r2).  hipcc's FP64 sqrt is
// rsq and three Newton-type corrections between a scaling of operands below
// 2^-767 and a selection for zero and infinity (read from this library's own
// assembly); its division is described in exact_div.hpp.  With r2 in
// [2^-190, 2^190) none of the scalings and selections applies to the root, and
// D^3 in [2^-285, 2^285] is inside the division's window.  A numerator is in
// it (or the zero of a zero separation or mass, for which the same operations give
// the zero `/` gives) when
//   - G m is zero or |G m| lies in [2^-100, 2^100), and
//   - every coordinate of both bodies is zero or at least 2^-140 in magnitude:
//     a difference of two such numbers is zero or at least 2^-193.
// Those two are checked once a body; r2 once a term.  A term outside takes
// sqrt and div3.  44 FP64 instructions against about 100 and five branches.
#pragma once
#include "exact_div.hpp"

#pragma clang fp contract(off)

namespace {

__device__ inline unsigned hi_word(double v)
{
    return (unsigned)((unsigned long long)__double_as_longlong(v) >> 32);
}

// |v| >= 2^-140; ok: or zero (infinities and NaN leave r2's window).
__device__ inline bool coord_big(double v)
{
    return (hi_word(v) & 0x7fffffffu) >= ((1023u - 140u) << 20);
}

__device__ inline bool coord_ok(double v) { return coord_big(v) || v == 0.0; }

// |G m| in [2^-100, 2^100); ok: or zero.  (With massless and negative ones outside
// the window, a field of 1000 such bodies took 17.0 to 19.0 us, 12.1 to 12.4 so.)
__device__ inline bool gm_big(double v)
{
    return (hi_word(v) & 0x7fffffffu) - ((1023u - 100u) << 20) < (200u << 20);
}

__device__ inline bool gm_ok(double v) { return gm_big(v) || v == 0.0; }

// r2 in [2^-190, 2^190).
__device__ inline bool r2_ok(double v)
{
    return hi_word(v) - ((1023u - 190u) << 20) < (380u << 20);
}

// The quotients n[c] / sqrt(r2)^3 (NEG: negated), in place, for operands in the
// window above.
template <bool NEG>
__device__ inline void window_quotients(double *n, double r2)
{
    double h = __builtin_amdgcn_rsq(r2);
    double g = r2 * h;
    h = h * 0.5;
    const double e = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, e, g);
    h = __builtin_fma(h, e, h);
    g = __builtin_fma(__builtin_fma(-g, g, r2), h, g);
    const double D = __builtin_fma(__builtin_fma(-g, g, r2), h, g);
    const double D3 = D * D * D;
    double y = __builtin_amdgcn_rcp(D3);
    y = __builtin_fma(y, __builtin_fma(-D3, y, 1.0), y);
    y = __builtin_fma(y, __builtin_fma(-D3, y, 1.0), y);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        // With r = n - D3 q, the quotient is r y + q and its negative -(r y + q),
        // the same rounding.  A zero n leaves r = 0, whose sign decides that of
        // the result: from fma(-D3, q, n) it is +0, which keeps the sign in -r y
        // - q, and from fma(D3, q, -n), there -r, it keeps the sign in r y + q.
        const double q = n[c] * y;
        if (NEG) n[c] = __builtin_fma(-__builtin_fma(-D3, q, n[c]), y, -q);
        else n[c] = __builtin_fma(-__builtin_fma(D3, q, -n[c]), y, q);
    }
}

}  // namespace
