// Device evaluation of one sphere pair in the reference's exact arithmetic.
//
// The reference computes every pair (A > B) in the body of its triangular loop,
// ColliderSingleCore/ColliderSingleCore.cpp:104-250 (and the same body in
// init_conditions, ball_group.hpp:784-936).  To be bitwise-equal to it on the
// GPU the device must perform the same IEEE binary64 operations in the same
// order: the expressions below keep the reference's evaluation order
// (left-to-right products, vec3 component order, norm = sqrt((x*x+y*y)+z*z),
// normalized = 3 divisions, vec3.hpp:44-128,180-184), the translation unit is
// compiled with -ffp-contract=off, and division and sqrt are the correctly
// rounded forms clang emits for binary64 on gfx950.
#pragma once

#include "sl_common.hpp"

#pragma clang fp contract(off)

namespace sl {

struct D3 {
    double x, y, z;
};

__device__ __forceinline__ D3 d3(double x, double y, double z) { return D3{x, y, z}; }
__device__ __forceinline__ D3 operator+(D3 a, D3 b) { return d3(a.x + b.x, a.y + b.y, a.z + b.z); }
__device__ __forceinline__ D3 operator-(D3 a, D3 b) { return d3(a.x - b.x, a.y - b.y, a.z - b.z); }
__device__ __forceinline__ D3 operator-(D3 a) { return d3(-a.x, -a.y, -a.z); }
// vector times scalar: the reference multiplies scalar * component (vec3.hpp:66)
__device__ __forceinline__ D3 operator*(D3 a, double s) { return d3(s * a.x, s * a.y, s * a.z); }
__device__ __forceinline__ D3 operator/(D3 a, double s) { return d3(a.x / s, a.y / s, a.z / s); }
__device__ __forceinline__ double dot(D3 a, D3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ double norm(D3 a) { return __builtin_sqrt(a.x * a.x + a.y * a.y + a.z * a.z); }
__device__ __forceinline__ D3 cross(D3 a, D3 b)
{
    return d3(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x);
}

// Magnitude factor of the vdW force at surface separation h, in the reference's
// product order: Ha/6*64*Ra*Ra*Ra*Rb*Rb*Rb*((h+Ra+Rb)/(s*s*t*t)),
// s = h^2 + 2Ra h + 2Rb h, t = s + 4 Ra Rb.
__device__ __forceinline__ double vdw_factor(double Ha, double Ra, double Rb, double h, double h2)
{
    const double twoRah = 2 * Ra * h;
    const double twoRbh = 2 * Rb * h;
    const double s = h2 + twoRah + twoRbh;
    const double t = h2 + twoRah + twoRbh + 4 * Ra * Rb;
    return Ha / 6 * 64 * Ra * Ra * Ra * Rb * Rb * Rb * ((h + Ra + Rb) / (s * s * t * t));
}

// vdW potential between spheres at surface separation h (ColliderSingleCore.cpp:195-202).
__device__ __forceinline__ double vdw_energy(double Ha, double Ra, double Rb, double S, double h)
{
    const double dR = Ra - Rb;
    const double z = S + h;
    const double two_RaRb = 2 * Ra * Rb;
    const double ds = z * z - (S * S);
    const double dd = z * z - (dR * dR);
    return -Ha / 6 * (two_RaRb / ds + two_RaRb / dd + ::log(ds / dd));
}

// a / b, correctly rounded, from y = RN(1/b), the correctly rounded reciprocal (one
// binary64 division per divisor): q0 = a y, then two corrections q <- q + (a - b q) y whose
// residual a - b q an FMA forms exactly.  The first correction leaves q within one ulp of
// a/b, so the second residual is exact and, y being within half an ulp of 1/b, the second
// correction rounds to the correctly rounded quotient (Markstein's theorem; P. Markstein,
// IBM J. Res. Dev. 34(1), 1990).  Valid while a, a/b and the residuals are normal numbers.
// A zero quotient can come out +0 where a / b gives -0; every use here adds it to a sum
// that started at +0, whose bits that does not change.
__device__ __forceinline__ double div_rcp(double a, double b, double y)
{
    const double q0 = a * y;
    const double q1 = __builtin_fma(__builtin_fma(-q0, b, a), y, q0);
    return __builtin_fma(__builtin_fma(-q1, b, a), y, q1);
}

// ---- square root and division without the special cases ---------------------------------
// For operands whose exponents (and their results') stay far inside binary64's range the
// compiler's square root and division spend a third of their instructions on scaling and
// special values.  These are the same iterations without those, for the far-field arm, which
// sends pairs outside FarRange to the general arm: bit for bit sqrt(x) and n / d.

// s = RN(sqrt(x)) by Goldschmidt's iteration from the hardware estimate (24 bits), two
// corrections by the FMA-exact residual x - s^2; y = RN(1/s) from the iteration's other half,
// h = 1/(2 sqrt x) to 46 bits, by two Newton steps (the first leaves y within an ulp, the
// residual 1 - s y of the second is exact; only a significand of all ones can come out one
// ulp off, where div_rcp's quotient is still right).
__device__ __forceinline__ void sqrt_rcp(double x, double& s, double& y)
{
    const double y0 = __builtin_amdgcn_rsq(x);
    const double g0 = x * y0, h0 = 0.5 * y0;
    const double r0 = __builtin_fma(-h0, g0, 0.5);
    const double g1 = __builtin_fma(g0, r0, g0), h1 = __builtin_fma(h0, r0, h0);
    const double g2 = __builtin_fma(__builtin_fma(-g1, g1, x), h1, g1);
    s = __builtin_fma(__builtin_fma(-g2, g2, x), h1, g2);
    const double y1 = h1 + h1;
    const double y2 = __builtin_fma(__builtin_fma(-s, y1, 1.0), y1, y1);
    y = __builtin_fma(__builtin_fma(-s, y2, 1.0), y2, y2);
}

// RN(n / d): two Newton steps on the hardware reciprocal, then Markstein's correction of the
// quotient by its FMA-exact residual.
__device__ __forceinline__ double div_plain(double n, double d)
{
    double y = __builtin_amdgcn_rcp(d);
    y = __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
    y = __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
    const double q = n * y;
    return __builtin_fma(__builtin_fma(-d, q, n), y, q);
}

// n / s^2 for the distance s and y = RN(1/s): 1/s^2 from y^2 (2 ulps) by one Newton step,
// which leaves it within 2^-48 of half an ulp of 1/s^2; div_rcp's quotient needs no more.
__device__ __forceinline__ double div_sq(double n, double s2, double y)
{
    const double z = y * y;
    return div_rcp(n, s2, __builtin_fma(__builtin_fma(-s2, z, 1.0), z, z));
}

// The range of the above: d^2 in [2^-200, 2^200) (checked pair by pair), radii and h_min in
// [2^-100, 2^100), masses in [2^-300, 2^300), G 0 or in [2^-100, 2^100).  Then s t of the far
// arm's denominator lies in 2^-400 .. 2^410, its square and every quotient and residual
// inside 2^+-910.
struct FarRange {
    __device__ static bool within(double x, int lo, int hi)   // 2^lo <= x < 2^hi
    {
        const unsigned e = (unsigned)(__double_as_longlong(x) >> 52);   // sign and exponent
        return e - (unsigned)(1023 + lo) < (unsigned)(hi - lo);
    }
    __device__ static bool ball(double R, double m) { return within(R, -100, 100) && within(m, -300, 300); }
    __device__ static bool params(const Phys& P) { return within(P.h_min, -100, 100) && (P.G == 0 || within(P.G, -100, 100)); }
    __device__ static bool distance2(double d2) { return within(d2, -200, 200); }
};

struct PairIn {
    D3 pA, pB;    // positions (after this step's drift)
    double RA, RB, mA, mB;
};

struct PairOut {
    D3 F;         // force on A
    D3 tA, tB;    // torques on A and B (touching pairs)
    double pe;    // pair energy (write steps)
    int contact;
};

// Previous full-step velocities and spins of a touching pair, and the separation of the
// positions the previous pair pass used.
struct TouchState {
    D3 vA, vB, wA, wB, q;
};

// pair_ref's touching arm (ColliderSingleCore.cpp:119-204) for a pair with overlap > 0,
// bit for bit, with the divisions by the distance, its square, S and the norms taken from one
// reciprocal each (div_rcp) and no second look at whether the pair touches: 520 instructions
// instead of 710, on the serial path of whoever waits for the pair.  Valid while every
// operand is normal: the caller checks FarRange for radii, masses and d^2; the components
// divided here may be 0 but not below 2^-700, and results must be finite.  Returns false
// where that does not hold (o is then to be taken from pair_ref).
__device__ __forceinline__ bool touch_pair_ref(const Phys& P, bool write, const PairIn& in, const TouchState& ts,
                                               PairOut& o)
{
    const double S = in.RA + in.RB;
    const D3 r = in.pB - in.pA;
    const double d2 = dot(r, r), q2 = dot(ts.q, ts.q);
    double dist, yd, old_dist, yq;
    sqrt_rcp(d2, dist, yd);
    sqrt_rcp(q2, old_dist, yq);
    const double overlap = S - dist;
    const double k = (dist >= old_dist) ? P.kout : P.kin;
    const double h = P.h_min, h2 = h * h;
    const double twoRah = 2 * in.RA * h, twoRbh = 2 * in.RB * h;
    const double sv = h2 + twoRah + twoRbh;
    const double tv = h2 + twoRah + twoRbh + 4 * in.RA * in.RB;
    const double fv = P.Ha / 6 * 64 * in.RA * in.RA * in.RA * in.RB * in.RB * in.RB *
                      div_plain(h + in.RA + in.RB, sv * sv * tv * tv);
    const D3 rh = d3(div_rcp(r.x, dist, yd), div_rcp(r.y, dist, yd), div_rcp(r.z, dist, yd));
    const double dd = dist * dist, z = yd * yd;
    const double ydd = __builtin_fma(__builtin_fma(-dd, z, 1.0), z, z);   // as in div_sq
    const D3 f_vdw = rh * fv;
    const D3 f_el = rh * (-k * overlap * .5);
    const D3 f_g = rh * div_rcp(P.G * in.mA * in.mB, dd, ydd);
    const double f_el_mag = norm(f_el);
    const double yS = div_plain(1.0, S);
    const D3 nA = r * in.RA, nB = (-r) * in.RB;
    const D3 r_a = d3(div_rcp(nA.x, S, yS), div_rcp(nA.y, S, yS), div_rcp(nA.z, S, yS));
    const D3 r_b = d3(div_rcp(nB.x, S, yS), div_rcp(nB.y, S, yS), div_rcp(nB.z, S, yS));
    const D3 w_diff = ts.wA - ts.wB;
    const D3 d_vel = ts.vB - ts.vA;
    const D3 rdd = d3(div_rcp(r.x, dd, ydd), div_rcp(r.y, dd, ydd), div_rcp(r.z, dd, ydd));
    const D3 v_rel = ((d_vel - rdd * dot(d_vel, r)) - cross(ts.wA, r_a)) - cross(ts.wB, r_a);
    auto exps = [](D3 a) {   // smallest exponent of the components (0 for a zero)
        return min(__builtin_amdgcn_frexp_exp(a.x), min(__builtin_amdgcn_frexp_exp(a.y), __builtin_amdgcn_frexp_exp(a.z)));
    };
    int e_min = min(exps(r), exps(v_rel));
    D3 slide = d3(0, 0, 0), roll = d3(0, 0, 0);
    const double v_rel_mag = norm(v_rel);
    if (v_rel_mag > 1e-13) {
        const double y = 1.0 / v_rel_mag;
        slide = d3(div_rcp(v_rel.x, v_rel_mag, y), div_rcp(v_rel.y, v_rel_mag, y), div_rcp(v_rel.z, v_rel_mag, y)) *
                (P.u_s * f_el_mag);
    }
    if (norm(w_diff) > 1e-13) {
        const D3 c = cross(w_diff, r_a);
        const D3 n = c * (-P.u_r * f_el_mag);
        const double cm = norm(c), y = 1.0 / cm;
        e_min = min(e_min, exps(n));
        roll = d3(div_rcp(n.x, cm, y), div_rcp(n.y, cm, y), div_rcp(n.z, cm, y));
    }
    o.F = ((f_g + f_el) + slide) + f_vdw;
    o.tA = cross(r_a, slide + roll);
    o.tB = cross(r_b, (-slide) + roll);
    o.pe = 0;
    if (write) {
        double pe = vdw_energy(P.Ha, in.RA, in.RB, S, h) + 0.5 * k * overlap * overlap;
        if (P.far_gravity) pe = pe + -P.G * in.mA * in.mB / dist;
        o.pe = pe;
    }
    o.contact = 1;
    const double all = ::fabs(o.F.x) + ::fabs(o.F.y) + ::fabs(o.F.z) + ::fabs(o.tA.x) + ::fabs(o.tA.y) + ::fabs(o.tA.z) +
                       ::fabs(o.tB.x) + ::fabs(o.tB.y) + ::fabs(o.tB.z);
    return e_min > -700 && FarRange::distance2(q2) && all < __builtin_huge_val();
}

// Full pair evaluation.  Velocities and spins are the previous full-step ones
// (the loop reads O.vel and O.w); they and old_dist are only read for touching
// pairs, through the callables, so the far-field arm loads nothing extra.
template <class ContactData>
__device__ __forceinline__ void pair_ref(const Phys& P, bool write, const PairIn& in,
                                         const ContactData& cd, PairOut& o)
{
    const double S = in.RA + in.RB;
    const D3 r = in.pB - in.pA;                   // vector from A to B
    const double dist = norm(r);
    const double overlap = S - dist;
    o.tA = d3(0, 0, 0);
    o.tB = d3(0, 0, 0);
    o.pe = 0;
    if (overlap > 0) {
        const double old_dist = cd.old_dist();
        const double k = (dist >= old_dist) ? P.kout : P.kin;   // :122-126
        const double h = P.h_min;                                // :129
        const double fv = vdw_factor(P.Ha, in.RA, in.RB, h, h * h);
        const D3 f_vdw = (r / norm(r)) * fv;                     // :135-139
        const D3 f_el = (r / dist) * (-k * overlap * .5);        // :142
        const D3 f_g = (r / dist) * (P.G * in.mA * in.mB / (dist * dist));  // :145
        const double f_el_mag = norm(f_el);                      // :154
        const D3 r_a = (r * in.RA) / S;                          // :155
        const D3 r_b = ((-r) * in.RB) / S;                       // :156
        const D3 wA = cd.wA(), wB = cd.wB();
        const D3 w_diff = wA - wB;                               // :157
        const D3 d_vel = cd.vB() - cd.vA();                      // :160
        // :161-162, the second spin term uses r_a as the reference writes it
        const D3 v_rel = ((d_vel - (r / (dist * dist)) * dot(d_vel, r)) - cross(wA, r_a)) - cross(wB, r_a);
        D3 slide = d3(0, 0, 0), roll = d3(0, 0, 0);
        const double v_rel_mag = norm(v_rel);
        if (v_rel_mag > 1e-13) slide = (v_rel / v_rel_mag) * (P.u_s * f_el_mag);       // :166-170
        const double w_diff_mag = norm(w_diff);
        if (w_diff_mag > 1e-13) {                                                   // :174-178
            const D3 c = cross(w_diff, r_a);
            roll = (c * (-P.u_r * f_el_mag)) / norm(c);
        }
        o.F = ((f_g + f_el) + slide) + f_vdw;                    // :181
        o.tA = cross(r_a, slide + roll);                         // :184
        o.tB = cross(r_b, (-slide) + roll);                      // :185
        if (write) {
            double pe = vdw_energy(P.Ha, in.RA, in.RB, S, h) + 0.5 * k * overlap * overlap;  // :195-203
            if (P.far_gravity) pe = pe + -P.G * in.mA * in.mB / dist;
            o.pe = pe;
        }
        o.contact = 1;
    } else {
        double h = ::fabs(overlap);                              // :211-215
        if (h < P.h_min) h = P.h_min;
        const double fv = vdw_factor(P.Ha, in.RA, in.RB, h, h * h);
        o.F = (r / norm(r)) * fv;                                // :221-227
        if (P.far_gravity) o.F = o.F + (r / dist) * (P.G * in.mA * in.mB / (dist * dist));
        if (write) {
            double pe = vdw_energy(P.Ha, in.RA, in.RB, S, h);    // :231-239
            if (P.far_gravity) pe = pe + -P.G * in.mA * in.mB / dist;
            o.pe = pe;
        }
        o.contact = 0;
    }
}

}  // namespace sl
