// Far-field pair algebra for the fast path.
//
// For a pair that is not touching and whose surface gap h = d - S is at least
// h_min (S = Ri + Rj, d = |r|), the reference's vdW force
//     F = Ha/6*64 Ri^3 Rj^3 (h+S)/(s^2 t^2) * r/d,   s = h^2+2(Ri+Rj)h, t = s+4RiRj
// (ColliderSingleCore.cpp:211-225) simplifies exactly, because h + S = d:
//     s = d^2 - (Ri+Rj)^2,   t = d^2 - (Ri-Rj)^2,   F = C_ij / (s^2 t^2) * r
// with C_ij = (Ha/6*64) Ri^3 Rj^3 = q_i q_j.  No square root is needed, and the
// pair is "near" (routed to the exact path) iff s < 2 S h_min + h_min^2.
// Gravity on all pairs is G m_i m_j r / d^3 = g_i g_j r * rsqrt(d^2)^3.
// The vdW energy of the same pair is U = -Ha/6 (2RiRj/s + 2RiRj/t + ln(s/t))
// (ColliderSingleCore.cpp:231-238 with z = S + h = d).
#pragma once

#include "sl_common.hpp"

namespace sl {

// 1/x: hardware reciprocal (24.4 good bits, measured over 4M operands spanning 2^+-60)
// and one Newton-Raphson step y <- y + y (1 - x y), 48.7 good bits (2.2e-15 relative):
// the size of the far-field algebra's other reassociation errors, far inside the
// fast path's 1e-13 force bar, for two FMAs less per pair than a second step.
#ifndef SL_RCP_NEWTON_STEPS
#define SL_RCP_NEWTON_STEPS 1
#endif
__device__ __forceinline__ double rcp_f64(double x)
{
    double y = __builtin_amdgcn_rcp(x);
    for (int k = 0; k < SL_RCP_NEWTON_STEPS; k++) {
        const double e = __builtin_fma(-x, y, 1.0);
        y = __builtin_fma(y, e, y);
    }
    return y;
}

// 1/sqrt(x): hardware estimate and one Newton step y <- y (3/2 - x/2 y^2), about
// 46 good bits; used only for the gravity term, which is many orders of magnitude
// below the vdW term inside a dust aggregate.
__device__ __forceinline__ double rsq_f64(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    const double hx = 0.5 * x;
    const double e = __builtin_fma(-hx * y, y, 0.5);
    return __builtin_fma(y, e, y);
}

// vdW energy of a far pair over -Ha/6, from s = d^2 - S^2, t = d^2 - (Ri-Rj)^2 (use: the lane's
// pair counts).  With y = 4 Ri Rj / t the reference's sum 2RiRj/s + 2RiRj/t + ln(s/t) is
// y/2/(1-y) + y/2 + ln(1-y) = sum over k >= 3 of (1/2 - 1/k) y^k: its first two orders
// cancel, so for y <= 1/8 (about three diameters apart and more: nearly every pair) 18 terms
// of the series give it to 2^-52, for 23 instructions, where the three divisions and the
// logarithm took about 75 and lost 6 / y^2 ulps.  (With the line at y = 1/16, 13 terms, the
// closed form's loss just above it was 2e-13 of a pair, and the sweep was no faster.)
// FAR: y <= 2^-5 for every pair of the tile (eleven radii apart), so 11 terms do (the first left
// out is 2.6 y^11 of the sum, 2^-53.6) and no lane needs the closed form.
// The write step's sweep at 40,000 spheres took 4557 us in the closed form, 2205 by 18 terms
// and 1890 with the short series (without energies: 1020); at 5,000 87, 55 and 54.
// energy_series: the sum to the term LAST, y and 1/t.
template <int LAST>
__device__ __forceinline__ double energy_series(double Ri, double Rj, double t, double& y, double& rt)
{
    rt = __builtin_amdgcn_rcp(t);
    rt = __builtin_fma(rt, __builtin_fma(-t, rt, 1.0), rt);
    rt = __builtin_fma(rt, __builtin_fma(-t, rt, 1.0), rt);
    y = 4 * Ri * Rj * rt;
    double p = 0.5 - 1.0 / LAST;
#pragma unroll
    for (int k = LAST - 1; k >= 3; k--) p = __builtin_fma(p, y, 0.5 - 1.0 / k);
    return p * (y * y * y);
}

template <bool FAR>
__device__ __forceinline__ double far_energy(double Ri, double Rj, double s, double t, bool use)
{
    double y, rt;
    if constexpr (FAR) return energy_series<13>(Ri, Rj, t, y, rt);
    double u = energy_series<20>(Ri, Rj, t, y, rt);
    const bool close = use && !(y <= 0.125);
    if (__any(close)) {
        const double q = s * rt;   // 1 - y, from s
        double rq = __builtin_amdgcn_rcp(q);
        rq = __builtin_fma(rq, __builtin_fma(-q, rq, 1.0), rq);
        rq = __builtin_fma(rq, __builtin_fma(-q, rq, 1.0), rq);
        const double v = __builtin_fma(0.5 * y, rq, 0.5 * y) + ::log(q);
        u = close ? v : u;
    }
    return u;
}

}  // namespace sl
