// Ordered-mode kernels: bitwise the reference's single-core arithmetic.
//
// The reference adds pair contributions into acc[i] and aacc[i] in ascending
// partner index j (its triangular loop visits (A=i, B<i) first, then (A>i, B=i),
// ColliderSingleCore.cpp:100-103).  Floating-point addition is not associative,
// so the GPU reproduces that order with one sequential accumulator per (ball,
// component), while the expensive part -- evaluating the pair -- runs on every
// lane (k_pairs_ordered below: a ring of wavefronts per group of balls, each evaluating
// a batch of partners and adding it when the sums reach it).
// Far pairs contribute +0.0 to aacc and j == i contributes +0.0 to both; an
// accumulator that starts at +0.0 under round-to-nearest never becomes -0.0,
// so these additions leave it bit-for-bit unchanged and are skipped.
//
// PE is summed per ball A over its partners B < A in ascending B, and the per-ball sums
// over A in ascending order by the caller: the same for every launch shape, but grouped
// per ball rather than the reference's single running sum, so it agrees to rounding only.
#include "sl_common.hpp"
#include "sl_fast_pair.hpp"
#include "sl_pair_ref.hpp"

#include <type_traits>

#pragma clang fp contract(off)

namespace sl {

namespace {

struct GlobalContact {
    const State& s;
    int A, B;
    __device__ D3 vA() const { return d3(s.f[VX][A], s.f[VY][A], s.f[VZ][A]); }
    __device__ D3 vB() const { return d3(s.f[VX][B], s.f[VY][B], s.f[VZ][B]); }
    __device__ D3 wA() const { return d3(s.f[WX][A], s.f[WY][A], s.f[WZ][A]); }
    __device__ D3 wB() const { return d3(s.f[WX][B], s.f[WY][B], s.f[WZ][B]); }
    // distance of the pair in the previous pair pass, recomputed from the
    // positions that pass used with the same operations (|x_B - x_A|)
    __device__ double old_dist() const
    {
        const D3 qa = d3(s.f[QX][A], s.f[QY][A], s.f[QZ][A]);
        const D3 qb = d3(s.f[QX][B], s.f[QY][B], s.f[QZ][B]);
        return norm(qb - qa);
    }
};

__device__ __forceinline__ D3 load3(const State& s, int f, int b) { return d3(s.f[f][b], s.f[f + 1][b], s.f[f + 2][b]); }

// Lanes of the mask below this one.
__device__ __forceinline__ int lanes_below(unsigned long long mask)
{
    return __builtin_popcountll(mask & ((1ull << (threadIdx.x % 64)) - 1));
}

template <int N>
__device__ __forceinline__ double block_sum(double v, double* red)
{
    // fixed-shape tree over the block: deterministic
    const int t = threadIdx.x;
    red[t] = v;
    __syncthreads();
    for (int s = N / 2; s > 0; s >>= 1) {
        if (t < s) red[t] = red[t] + red[t + s];
        __syncthreads();
    }
    const double r = red[0];
    __syncthreads();
    return r;
}

}  // namespace

// First pass (ColliderSingleCore.cpp:82-97) plus the hysteresis state: the
// positions before the drift are the ones the previous pair pass used.  To d: the state
// itself, or (COPY) another set, with the velocities and spins the step will read.
template <bool COPY>
__global__ void k_drift(State s, State d, int n, double dt)
{
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= n) return;
    const double px = s.f[PX][b], py = s.f[PY][b], pz = s.f[PZ][b];
    if (COPY)
        for (int f = VX; f < VX + 6; f++) d.f[f][b] = s.f[f][b];
    d.f[QX][b] = px;
    d.f[QY][b] = py;
    d.f[QZ][b] = pz;
    const double hx = s.f[VX][b] + .5 * s.f[AX][b] * dt;
    const double hy = s.f[VY][b] + .5 * s.f[AY][b] * dt;
    const double hz = s.f[VZ][b] + .5 * s.f[AZ][b] * dt;
    d.f[HX][b] = hx;
    d.f[HY][b] = hy;
    d.f[HZ][b] = hz;
    d.f[GX][b] = s.f[WX][b] + .5 * s.f[BX][b] * dt;
    d.f[GY][b] = s.f[WY][b] + .5 * s.f[BY][b] * dt;
    d.f[GZ][b] = s.f[WZ][b] + .5 * s.f[BZ][b] * dt;
    d.f[PX][b] = px + hx * dt;
    d.f[PY][b] = py + hy * dt;
    d.f[PZ][b] = pz + hz * dt;
}

// Positions the step-0 pass uses are also its hysteresis reference (k = kout
// for a pair overlapping at step 0).
__global__ void k_copy_prev(State s, int n)
{
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= n) return;
    s.f[QX][b] = s.f[PX][b];
    s.f[QY][b] = s.f[PY][b];
    s.f[QZ][b] = s.f[PZ][b];
}

// One pair (i, j) in the reference's arithmetic, touching or not (ColliderSingleCore.cpp:
// 119-250), in its orientation A = max(i, j): ball i's acc contribution to c3[0], c3[cs],
// c3[2 cs], its aacc contribution to a3[0], a3[as], a3[2 as], and the pair energy (write
// steps, i = A) to *pe.  Returns 1 for a touching pair.
__device__ __forceinline__ int general_pair(const State& s, const Phys& P, int write, int i, int j, double ymi, double* c3,
                                            int cs, double* a3, int as, double* pe)
{
    const bool iA = i > j;
    const D3 pi = d3(s.f[PX][i], s.f[PY][i], s.f[PZ][i]);
    const D3 pj = d3(s.f[PX][j], s.f[PY][j], s.f[PZ][j]);
    const double Ri = s.f[RAD][i], mi = s.f[MASS][i], Ii = s.f[MOI][i];
    const double Rj = s.f[RAD][j], mj = s.f[MASS][j];
    PairIn in;
    in.pA = iA ? pi : pj;
    in.pB = iA ? pj : pi;
    in.RA = iA ? Ri : Rj;
    in.RB = iA ? Rj : Ri;
    in.mA = iA ? mi : mj;
    in.mB = iA ? mj : mi;
    PairOut o;
    GlobalContact gcx{s, iA ? i : j, iA ? j : i};
    pair_ref(P, write && iA, in, gcx, o);
    // acc[A] += F/m[A] or acc[B] -= F/m[B]; aacc[A] += tA/moi[A], aacc[B] += tB/moi[B] (:187-188, 249-250)
    D3 a = d3(div_rcp(o.F.x, mi, ymi), div_rcp(o.F.y, mi, ymi), div_rcp(o.F.z, mi, ymi));
    if (!iA) a = -a;
    const D3 aa = (iA ? o.tA : o.tB) / Ii;
    c3[0] = a.x;
    c3[cs] = a.y;
    c3[2 * cs] = a.z;
    a3[0] = aa.x;
    a3[as] = aa.y;
    a3[2 * as] = aa.z;
    *pe = iA ? o.pe : 0.0;
    return o.contact;
}

// A partner's position, radius, mass and Ha/6*64 R^3 (the first factors of the vdW prefactor
// when the partner is A) as the far-field arm reads them (48 bytes: three 16-byte LDS reads).
struct PartnerRec {
    double x, y, z, R, m, pref;
};

// A ball of the workgroup: position, radius, mass, 1/m (divisions by m through div_rcp) and its
// factors of the reference's products when it is A (Ha/6*64 Ra^3, G mA).
struct BallRec {
    double x, y, z, R, m, ym, pref, Gm;
};

// The pair pass as a ring of wavefronts.  A workgroup owns NB balls and its W wavefronts take
// the partners in batches of BP = CH * 64/NB, batch m by wavefront m mod W:
//   evaluate  lane (ball l % NB, slot l / NB) evaluates CH pairs of its ball, one per step q,
//             by the far-field arm in the reference orientation and writes the ball's signed
//             acc contribution to the wavefront's own LDS buffer.  Lanes whose pair touches
//             are noted by step; what the far arm wrote for them is replaced before it is
//             added.
//   add       when the running sums have passed through every earlier batch (turn == m), one
//             lane per (ball, component) adds its BP contributions in ascending j and hands
//             the sums on.  aacc gets only the touching pairs' contributions: the others are
//             +0.0, a no-op on a sum that starts at +0.0.
// Only the adding is serial (6.5 cycles a partner), and only the wavefront whose turn
// it is takes part in it: the others go on evaluating, with no barrier anywhere.  Every
// sum has the same order whatever the shape, so all launch shapes give the same bits (the
// energies included: per-ball sums, added over the balls in ascending order by the caller).
// Every wavefront of a workgroup is resident, and the owner of the batch whose turn it is
// waits for nothing but the contact table's maker, which waits for nothing: every wait ends.
// LDS instructions of a wavefront take effect in their order, which is all the handing on
// needs: sums, then turn; turn, then sums.
//
// Touching pairs.  The contact arm is five times the far arm's instructions, for one or two
// lanes of a wavefront, so a batch's touching pairs are numbered and evaluated side by side, up
// to 64 at a time, before the turn (64 AD of them: beyond, ab is used again and the turn has to
// come first).  Evaluated step by step, by the lanes that met them, and after the first AD steps
// within the turn, a ball with a thousand contacts took 180 us a step at 1,000 balls and 836 at
// 5,000; now 43 and 157, and 129 ordinary balls 8.3 instead of 9.7, 1,000 18.2 instead of 19.3.
// With SCAN the workgroup first tests its balls against every partner
// (16 instructions a step), and one wavefront evaluates the touching pairs found, up to
// 64, side by side while the others start on their batches; a pair met in the sweep is then
// copied from that table.  Pairs that did not fit in it, and all touching pairs without SCAN,
// are evaluated in their batch.  The scan
// pays up to about 1,700 balls (4 balls, 4 wavefronts, us per step with / without: 1,500 balls
// 35.1 / 37.1, 1,800 42.9 / 42.6, 2,200 58.9 / 54.9, 5,000 181 / 161): its cost grows with the
// partners, what it saves only with the contacts.
// While contacts are evaluated a lane's own ball waits in LDS (BallRec): in registers it took
// 26 spills more, the next batch's partners among them, which then had to arrive first.
//
// Bound by the binary64 pipe: 131 VALU instructions a step of 64 evaluations (105 of them the
// reference's arithmetic), 165 with the staging, the adding and the contacts; at 15,039
// balls that is 75% of the time, at 5,000 63% (1,250 workgroups, 3 to a CU).  Small systems are
// bound by the chain of adds (about 400 cycles a batch of 64) and by the first
// contacts' 5,000 cycles.  Measured per step, before (chunks of partners, a barrier each,
// sums by a wavefront of its own, the kick in a launch of its own) and now: 129 balls 16.5 ->
// 8.3 us, 1,000 29 -> 18.2, 2,200 87 -> 54.5, 5,000 259 -> 161, 15,039 1,750 -> 1,095.
//
// Write steps take a far pair's energy from the series (y <= 1/8; the logarithm and three
// divisions cost two thirds of a step more, and spilled up to 72 registers) and two wavefronts
// per SIMD: 15,039 balls 1,894 -> 1,584-1,720 us, 5,000 269 -> 238.
//
// With a second set of arrays (os.nxt) the owner of the last batch also kicks its balls and,
// with os.drift, drifts them into the next step (the operations of k_kick and k_drift): one
// launch a step instead of two.  The other workgroups may still be reading this step's positions and
// velocities, hence the second set.
struct OrdState {
    double* cur;           // dynamic fields, field f at cur + f stride
    const double* konst;   // radii, masses, moments of inertia, likewise (RAD ..)
    double* nxt;           // where the state after the step goes, or NULL: only acc and aacc, in place
    long stride;
    int drift;
    int* nonfinite;
};

template <int NB, int CH, int W, int AD, int WPE, int UNR, bool SCAN, bool WRITE>
__global__ __launch_bounds__(W * 64) __attribute__((amdgpu_waves_per_eu(WRITE && WPE > 2 ? 2 : WPE)))
void k_pairs_ordered(OrdState os, Phys P, int n, double* __restrict__ pe_ball,
                     unsigned long long* __restrict__ contacts)
{
    State s;
    for (int f = 0; f < NFIELD; f++) s.f[f] = (f < RAD ? os.cur : const_cast<double*>(os.konst)) + f * os.stride;
    constexpr int JS = 64 / NB;             // partners a wavefront evaluates at once
    constexpr int BP = CH * JS;             // partners per batch
    constexpr int NQ = WRITE ? 4 : 3;       // acc xyz, pair energy
    // A ball's contributions lie in a row, so that an adding lane reads two at once.  Row and
    // component strides: 16 lanes' stores (16/NB slots of NB balls) and 8 adding lanes' 16-byte
    // reads each cover the 32 banks once (65 thousand conflict cycles a launch at 5,000 balls;
    // 4.8 million when the stores were spread for 32 lanes and 64 banks, in the same time).
    constexpr int RS = (BP + 31) / 32 * 32 + 16 / NB, CS = NB * RS + 2;
    constexpr int AH = BP < 16 ? BP : 16;   // contributions a lane adds from registers at once
    static_assert(64 % NB == 0 && BP <= 64 && NQ * NB <= 64 && BP % AH == 0 && CH <= 4, "batch shape");
    __shared__ __attribute__((aligned(16))) double cb[W][NQ][CS];   // acc contributions (and energies)
    constexpr int AE = 64 * AD;             // touching pairs of a batch evaluated before its turn
    __shared__ double ab[W][3][AE];         // their aacc contributions, by number
    __shared__ unsigned char numbered[W][AE];   // their step << 6 | lane
    __shared__ PartnerRec sp[W][BP];
    __shared__ BallRec ball[NB];
    __shared__ double run[7][NB];           // the sums: acc xyz, aacc xyz, energy
    __shared__ double own[3][3][NB];        // half-step velocities and spins, positions: for the kick and the drift
    __shared__ int turn, ready, found;
    __shared__ unsigned ccount;
    __shared__ unsigned tkey[SCAN ? 64 : 1];        // contact table: ball << 24 | partner ...
    __shared__ double tres[SCAN ? 64 : 1][7];       // ... acc xyz, aacc xyz, energy

    const int t = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(t / 64), l = t % 64;
    for (int e = t; e < 7 * NB; e += 64 * W) (&run[0][0])[e] = 0.0;
    if (!WRITE && os.nxt && t < 3 * NB && (int)blockIdx.x * NB + t % NB < n) {
        const long e = t / NB * os.stride + blockIdx.x * NB + t % NB;
        (&own[0][0][0])[t] = os.cur[HX * os.stride + e];
        (&own[1][0][0])[t] = os.cur[GX * os.stride + e];
        (&own[2][0][0])[t] = os.cur[PX * os.stride + e];
    }
    if (t == 0) {
        turn = 0;
        ready = 0;
        found = 0;
        ccount = 0;
    }

    const int il = l % NB, jq = l / NB;
    const int i0 = blockIdx.x * NB, i = i0 + il;
    const bool iv = i < n;
    const double Hc = P.Ha / 6 * 64;
    if (t < NB) {
        const int b = i0 + t < n ? i0 + t : 0;
        const double R = s.f[RAD][b], mass = s.f[MASS][b];
        ball[t] = BallRec{s.f[PX][b], s.f[PY][b], s.f[PZ][b], R, mass, 1.0 / mass, Hc * R * R * R, P.G * mass};
    }
    unsigned cnt = 0;

    const int nm = (n + BP - 1) / BP;        // batches
    PartnerRec nx;                           // this lane's partner of the wavefront's next batch
    auto load_batch = [&](int m) {
        const int j = m * BP + l;
        if (l < BP && j < n)
            nx = PartnerRec{s.f[PX][j], s.f[PY][j], s.f[PZ][j], s.f[RAD][j], s.f[MASS][j], 0.0};
    };
    load_batch(w);
    __syncthreads();
    // Pair (ball bl of the workgroup, partner j) in full, by the touching arm where it holds: acc
    // and aacc contributions to c3[0], c3[cs], .. and a3[0], a3[as], ..; returns 1 if it touches.
    auto contact = [&](int bl, int j, double* c3, int cs, double* a3, int as, double* pe) -> int {
        const int bi = i0 + bl;
        const D3 pb = d3(ball[bl].x, ball[bl].y, ball[bl].z);
        const double Rb = ball[bl].R, mb = ball[bl].m, ymb = ball[bl].ym;
        const bool iA = bi > j;
        const D3 pj = d3(s.f[PX][j], s.f[PY][j], s.f[PZ][j]);
        const double Rj = s.f[RAD][j], mj = s.f[MASS][j];
        const D3 d = pj - pb;
        // (a scanned pair may not touch, nor one met beside a ball out of range)
        bool ok = FarRange::params(P) && FarRange::ball(Rb, mb) && FarRange::ball(Rj, mj) &&
                  FarRange::distance2(dot(d, d)) && (Rb + Rj) - norm(d) > 0;
        if (ok) {
            const int A = iA ? bi : j, B = iA ? j : bi;
            const TouchState ts{load3(s, VX, A), load3(s, VX, B), load3(s, WX, A), load3(s, WX, B),
                                load3(s, QX, B) - load3(s, QX, A)};
            const double Ib = s.f[MOI][bi];
            const PairIn in{iA ? pb : pj, iA ? pj : pb, iA ? Rb : Rj, iA ? Rj : Rb, iA ? mb : mj, iA ? mj : mb};
            PairOut o;
            ok = touch_pair_ref(P, WRITE && iA, in, ts, o);
            // acc[A] += F/m[A] or acc[B] -= F/m[B]; aacc[A] += tA/moi[A], aacc[B] += tB/moi[B]
            const D3 a = d3(div_rcp(o.F.x, mb, ymb), div_rcp(o.F.y, mb, ymb), div_rcp(o.F.z, mb, ymb));
            const D3 aa = (iA ? o.tA : o.tB) / Ib;
            c3[0] = iA ? a.x : -a.x;
            c3[cs] = iA ? a.y : -a.y;
            c3[2 * cs] = iA ? a.z : -a.z;
            a3[0] = aa.x;
            a3[as] = aa.y;
            a3[2 * as] = aa.z;
            *pe = o.pe;
        }
        if (ok) return 1;
        return general_pair(s, P, WRITE, bi, j, ymb, c3, cs, a3, as, pe);
    };

    unsigned mykey = ~0u;     // SCAN: the table's keys, one per lane, once read
    if constexpr (SCAN) {
        // every wavefront scans every W-th group of JS partners; a superset of the touching
        // pairs (d^2 against S^2, a little enlarged)
        constexpr int SU = 4;   // groups whose loads are in flight together
        const D3 pi = d3(ball[il].x, ball[il].y, ball[il].z);
        const double Ri = ball[il].R;
        for (int j1 = w * JS + jq; j1 - jq < n; j1 += SU * W * JS) {
            D3 pj[SU];
            double Rj[SU];
#pragma unroll
            for (int u = 0; u < SU; u++) {
                const int j = min(j1 + u * W * JS, n - 1);
                pj[u] = d3(s.f[PX][j], s.f[PY][j], s.f[PZ][j]);
                Rj[u] = s.f[RAD][j];
            }
#pragma unroll
            for (int u = 0; u < SU; u++) {
                const int j = j1 + u * W * JS;
                const D3 d = pj[u] - pi;
                const double S = Ri + Rj[u];
                if (dot(d, d) < S * S * (1 + 1e-12) && iv && j < n && j != i) {
                    const int e = atomicAdd(&found, 1);
                    if (e < 64) tkey[e] = (unsigned)il << 24 | (unsigned)j;
                }
            }
        }
        __syncthreads();
        const int nt = min(found, 64);
        if (w == W - 1) {
            __builtin_amdgcn_s_setprio(3);
            if (l < nt) {
                const unsigned key = tkey[l];
                double pe = 0;
                const int touch = contact((int)(key >> 24), (int)(key & 0xffffffu), &tres[l][0], 1, &tres[l][3], 1, &pe);
                if (WRITE) tres[l][6] = pe;
                if (!touch) tkey[l] = ~0u;
            }
            __builtin_amdgcn_s_setprio(0);
            asm volatile("" ::: "memory");
            if (l == 0) __hip_atomic_store(&ready, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
    }
    bool have_table = false;
    const bool gen_i = !FarRange::params(P) || !FarRange::ball(ball[il].R, ball[il].m);
    // this lane's ball, read again after contacts, which have its registers meanwhile
    D3 pi;
    double Ri, mi, ymi, prefA, Gmi, two_Ri, four_Ri;
    auto load_ball = [&]() {
        const BallRec& b = ball[il];
        pi = d3(b.x, b.y, b.z);
        Ri = b.R;
        mi = b.m;
        ymi = b.ym;
        prefA = b.pref;
        Gmi = b.Gm;
        two_Ri = 2 * Ri;
        four_Ri = 4 * Ri;
    };
    load_ball();

#pragma unroll 1
    for (int m = w; m < nm; m += W) {
        const int j0 = m * BP;
        // the batch's partners to LDS, the next batch's on their way
        bool bad = false;
        if (l < BP && j0 + l < n) {
            bad = !FarRange::ball(nx.R, nx.m);
            nx.pref = Hc * nx.R * nx.R * nx.R;
            sp[w][l] = nx;
        }
        const bool gen = gen_i || __any(bad);
        if (m + W < nm) load_batch(m + W);
        asm volatile("" ::: "memory");

        // steps whose pair touches or has operands outside FarRange: replaced after the sweep
        unsigned pend = 0;
        // One far-field pair (i, j) in the reference's orientation A = max(i, j): ball i
        // is A when IA (ColliderSingleCore.cpp:104-110, 211-227).  Writes ball i's acc
        // contribution (and its energy on write steps).
        auto far_pair = [&](auto ia, auto checked, int q) {
            constexpr bool IA = decltype(ia)::value;
            constexpr bool CHK = decltype(checked)::value;
            const int jl = jq + JS * q;
            const int j = j0 + jl;
            const bool pair = !CHK || (iv && j < n && j != i);
            const PartnerRec& pr = sp[w][jl];
            const D3 pj = d3(pr.x, pr.y, pr.z);
            const double Rj = pr.R, mj = pr.m;
            const double S = IA ? Ri + Rj : Rj + Ri;
            const D3 r = IA ? pj - pi : pi - pj;               // x_B - x_A
            const double d2 = dot(r, r);
            double dist, yd;                                   // norm(r) and its reciprocal
            sqrt_rcp(d2, dist, yd);
            const double overlap = S - dist;
            if (pair && (overlap > 0 || gen || !FarRange::distance2(d2))) pend |= 1u << q;
            double h = ::fabs(overlap);
            if (h < P.h_min) h = P.h_min;
            const double h2 = h * h;
            // vdw_factor with Ra = R_A, Rb = R_B: 2 Ra h, 2 Rb h, 4 Ra Rb and
            // Ha/6*64 Ra Ra Ra Rb Rb Rb in the reference's product order
            const double twoRah = IA ? two_Ri * h : (2 * Rj) * h;
            const double twoRbh = IA ? (2 * Rj) * h : two_Ri * h;
            const double sv = h2 + twoRah + twoRbh;
            const double tv = sv + (IA ? four_Ri * Rj : (4 * Rj) * Ri);
            const double quot = div_plain(IA ? h + Ri + Rj : h + Rj + Ri, sv * sv * tv * tv);
            const double fv = IA ? prefA * Rj * Rj * Rj * quot : pr.pref * Ri * Ri * Ri * quot;
            const D3 rh = d3(div_rcp(r.x, dist, yd), div_rcp(r.y, dist, yd), div_rcp(r.z, dist, yd));
            D3 F = rh * fv;
            if (P.far_gravity) F = F + rh * div_sq(IA ? Gmi * mj : P.G * mj * mi, dist * dist, yd);
            // acc[A] += F/m[A]  or  acc[B] -= F/m[B]   (:187-188, 249-250)
            double c0 = div_rcp(F.x, mi, ymi), c1 = div_rcp(F.y, mi, ymi), c2 = div_rcp(F.z, mi, ymi);
            double u = 0;
            if (WRITE && IA) {                                 // :228-240
                double y, rt;
                u = -P.Ha / 6 * energy_series<20>(Ri, Rj, tv, y, rt);
                const bool close = pair && !(y <= 0.125);
                if (__any(close)) {
                    const double v = vdw_energy(P.Ha, Ri, Rj, S, h);
                    u = close ? v : u;
                }
                if (P.far_gravity) u = u + div_rcp(-P.G * mi * mj, dist, yd);
            }
            if (CHK && !pair) c0 = c1 = c2 = u = 0;            // no partner, or the ball itself
            const int o_ = il * RS + jl;
            cb[w][0][o_] = IA ? c0 : -c0;
            cb[w][1][o_] = IA ? c1 : -c1;
            cb[w][2][o_] = IA ? c2 : -c2;
            if (WRITE) cb[w][NQ - 1][o_] = u;
        };
        if (j0 + BP <= i0 && i0 + NB <= n) {
            // every partner of the batch precedes every ball of the workgroup: i is A
#pragma unroll UNR
            for (int q = 0; q < CH; q++) far_pair(std::true_type{}, std::false_type{}, q);
        } else if (j0 >= i0 + NB && j0 + BP <= n) {
            // every partner follows: i is B
#pragma unroll UNR
            for (int q = 0; q < CH; q++) far_pair(std::false_type{}, std::false_type{}, q);
        } else {
#pragma unroll 1
            for (int q = 0; q < CH; q++) {
                if (i > j0 + jq + JS * q)
                    far_pair(std::true_type{}, std::true_type{}, q);
                else
                    far_pair(std::false_type{}, std::true_type{}, q);
            }
        }
        asm volatile("" ::: "memory");

        __builtin_amdgcn_s_setprio(3);
        auto get_table = [&]() {
            if (!have_table) {
                while (!__builtin_amdgcn_readfirstlane(__hip_atomic_load(&ready, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP))) {
                }
                asm volatile("" ::: "memory");
                if (l < min(found, 64)) mykey = tkey[l];
                have_table = true;
            }
        };
        const bool adds = l < NQ * NB;
        const int comp = adds ? jq : 0;
        double* const pr = &run[comp < 3 ? comp : 6][il];
        double r;
        auto wait_turn = [&]() {
            for (;;) {
                const int now = __hip_atomic_load(&turn, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                asm volatile("" ::: "memory");
                r = __hip_atomic_load(pr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);   // read after turn
                if (__builtin_amdgcn_readfirstlane(now) == m) break;
            }
            asm volatile("" ::: "memory");
        };
        // The batch's touching pairs, numbered ball by ball, j ascending.
        int first = 0, own_pairs = 0, pairs = 0;   // this lane's ball's first number, its pairs; all pairs
        const unsigned long long own_lanes = (~0ull / ((1ull << NB) - 1)) << il;   // lanes of this lane's ball
        auto number_pairs = [&]() {
#pragma unroll
            for (int q = 0; q < CH; q++) own_pairs += __builtin_popcountll(__ballot((pend >> q) & 1u) & own_lanes);
#pragma unroll
            for (int b = 0; b < NB; b++) {
                const int c = __builtin_amdgcn_readlane(own_pairs, b);   // lane b's ball is b
                if (b < il) first += c;
                pairs += c;
            }
        };
        // Contributions of pairs e0 .. e0 + AE - 1 to cb and ab, from the contact table or evaluated.
        auto fill_pairs = [&](int e0) {
            int e = first - e0;
#pragma unroll 1
            for (int q = 0; q < CH; q++) {
                const bool mine = (pend >> q) & 1u;
                const unsigned long long lanes = __ballot(mine) & own_lanes;
                const int at = e + lanes_below(lanes);
                if (mine && at >= 0 && at < AE) numbered[w][at] = (unsigned char)(q << 6 | l);
                e += __popcll(lanes);
            }
            asm volatile("" ::: "memory");
            const int m1 = min(pairs - e0, AE);
#pragma unroll 1
            for (int r0 = 0; r0 < m1; r0 += 64) {
                const int at = min(r0 + l, m1 - 1);
                const int z = numbered[w][at];
                const int bl = (z & 63) % NB, jl = JS * (z >> 6) + (z & 63) / NB, bi = i0 + bl, j = j0 + jl;
                double* const c3 = &cb[w][0][bl * RS + jl];
                double* const a3 = &ab[w][0][0] + at;
                bool mine = r0 + l < m1;
                if constexpr (SCAN) {
                    get_table();
                    const unsigned key = (unsigned)bl << 24 | (unsigned)j;
                    int te = -1;
                    for (int k = 0; k < min(found, 64); k++) te = (unsigned)__builtin_amdgcn_readlane(mykey, k) == key ? k : te;
                    if (mine && te >= 0) {
                        for (int k = 0; k < 3; k++) {
                            c3[k * CS] = tres[te][k];
                            a3[k * AE] = tres[te][3 + k];
                        }
                        if (WRITE) cb[w][NQ - 1][bl * RS + jl] = tres[te][6];
                        if (bi > j) cnt++;
                        mine = false;
                    }
                }
                if (mine) {
                    double pe = 0;
                    const int touch = contact(bl, j, c3, CS, a3, AE, &pe);
                    if (WRITE) cb[w][NQ - 1][bl * RS + jl] = pe;
                    if (touch && bi > j) cnt++;
                }
            }
            asm volatile("" ::: "memory");
        };
        // Theirs to aacc: the lane's ball's, in order.
        auto add_aacc = [&](int e0) {
            if (comp < 3 && adds) {
                double ra = run[3 + comp][il];
                const double* src = &ab[w][0][0] + comp * AE;
                const int e1 = min(first + own_pairs - e0, AE);
#pragma unroll 4
                for (int e = max(first - e0, 0); e < e1; e++) ra = ra + src[e];
                run[3 + comp][il] = ra;
            }
            asm volatile("" ::: "memory");
        };
        int last = 0;                       // those in ab: AE from here
        if (__any(pend != 0)) {
            number_pairs();
#pragma unroll 1
            for (; ; last += AE) {
                fill_pairs(last);
                if (last + AE >= pairs) break;
                wait_turn();                // ab is used again: these sums' turn has to come first
                add_aacc(last);
            }
            load_ball();
        }
        // add: lane (ball l % NB, component l / NB)
        if (adds) {
            typedef double double2_t __attribute__((ext_vector_type(2)));
            const double2_t* src = reinterpret_cast<const double2_t*>(&cb[w][comp][il * RS]);
            double2_t v[AH / 2];
#pragma unroll
            for (int q = 0; q < AH / 2; q++) v[q] = src[q];
            wait_turn();
#pragma unroll
            for (int q0 = 0; q0 < BP; q0 += AH) {
                double2_t u[AH / 2];
                if (q0 + AH < BP) {
#pragma unroll
                    for (int q = 0; q < AH / 2; q++) u[q] = src[(q0 + AH) / 2 + q];
                }
#pragma unroll
                for (int q = 0; q < AH / 2; q++) r = (r + v[q].x) + v[q].y;
                if (q0 + AH < BP) {
#pragma unroll
                    for (int q = 0; q < AH / 2; q++) v[q] = u[q];
                }
            }
            *pr = r;
        }
        if (pairs) add_aacc(last);
        asm volatile("" ::: "memory");
        if (l == 0) __hip_atomic_store(&turn, m + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (m == nm - 1 && adds && iv) {
            if (comp == 3) {
                pe_ball[i] = r;
            } else {
                const double al = run[3 + comp][il];
                const long c0 = comp * os.stride + i;
                auto at = [&](double* base, int f) -> double& { return base[f * os.stride + c0]; };
                if (WRITE || !os.nxt) {
                    at(os.cur, AX) = r;
                    at(os.cur, BX) = al;
                } else {
                    // closing kick (ColliderSingleCore.cpp:263-287)
                    const double dt = P.dt;
                    const double h0 = own[0][comp][il], g0 = own[1][comp][il], p0 = own[2][comp][il];
                    const double v = h0 + .5 * r * dt;
                    const double wv = g0 + .5 * al * dt;
                    if (!(isfinite(v) && isfinite(wv) && isfinite(p0))) atomicOr(os.nonfinite, 1);
                    at(os.nxt, VX) = v;
                    at(os.nxt, WX) = wv;
                    at(os.nxt, AX) = r;
                    at(os.nxt, BX) = al;
                    if (os.drift) {   // of the next step (:82-97)
                        const double hx = v + .5 * r * dt;
                        at(os.nxt, HX) = hx;
                        at(os.nxt, GX) = wv + .5 * al * dt;
                        at(os.nxt, QX) = p0;
                        at(os.nxt, PX) = p0 + hx * dt;
                    } else {
                        at(os.nxt, HX) = h0;
                        at(os.nxt, GX) = g0;
                        at(os.nxt, QX) = at(os.cur, QX);
                        at(os.nxt, PX) = p0;
                    }
                }
            }
        }
        __builtin_amdgcn_s_setprio(0);
        asm volatile("" ::: "memory");
    }

    // contact count (integer, order-independent)
    if (cnt) atomicAdd(&ccount, cnt);
    __syncthreads();
    // contacts[0]: the running total; contacts[1]: this write step's touching pairs
    if (t == 0 && ccount) {
        atomicAdd(contacts, (unsigned long long)ccount);
        if (WRITE) atomicAdd(contacts + 1, (unsigned long long)ccount);
    }
}

// Third pass (ColliderSingleCore.cpp:263-287): closing half kick and, on write
// steps, per-block partial sums of KE, momentum and angular momentum.
__global__ __launch_bounds__(256) void k_kick(State s, int n, double dt, int write, int kick,
                                              double* __restrict__ e_part,
                                              int* __restrict__ nonfinite)
{
    __shared__ double red[256];
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    double e[7] = {0, 0, 0, 0, 0, 0, 0};
    if (b < n) {
        double vx, vy, vz, wx, wy, wz;
        if (kick) {
            vx = s.f[HX][b] + .5 * s.f[AX][b] * dt;
            vy = s.f[HY][b] + .5 * s.f[AY][b] * dt;
            vz = s.f[HZ][b] + .5 * s.f[AZ][b] * dt;
            wx = s.f[GX][b] + .5 * s.f[BX][b] * dt;
            wy = s.f[GY][b] + .5 * s.f[BY][b] * dt;
            wz = s.f[GZ][b] + .5 * s.f[BZ][b] * dt;
            s.f[VX][b] = vx;
            s.f[VY][b] = vy;
            s.f[VZ][b] = vz;
            s.f[WX][b] = wx;
            s.f[WY][b] = wy;
            s.f[WZ][b] = wz;
        } else {
            vx = s.f[VX][b]; vy = s.f[VY][b]; vz = s.f[VZ][b];
            wx = s.f[WX][b]; wy = s.f[WY][b]; wz = s.f[WZ][b];
        }
        const double px = s.f[PX][b], py = s.f[PY][b], pz = s.f[PZ][b];
        if (!(isfinite(vx) && isfinite(vy) && isfinite(vz) && isfinite(wx) && isfinite(wy) &&
              isfinite(wz) && isfinite(px) && isfinite(py) && isfinite(pz)))
            atomicOr(nonfinite, 1);
        if (write) {
            const double m = s.f[MASS][b], I = s.f[MOI][b];
            const D3 v = d3(vx, vy, vz), w = d3(wx, wy, wz), p = d3(px, py, pz);
            e[0] = .5 * m * dot(v, v) + .5 * I * dot(w, w);      // :282-283
            const D3 mv = v * m;                                   // :284
            e[1] = mv.x; e[2] = mv.y; e[3] = mv.z;
            const D3 L = cross(p, v) * m + w * I;                  // :285
            e[4] = L.x; e[5] = L.y; e[6] = L.z;
        }
    }
    if (write) {
        for (int c = 0; c < 7; c++) {
            const double tot = block_sum<256>(e[c], red);
            if (threadIdx.x == 0) e_part[blockIdx.x * 7 + c] = tot;
        }
    }
}

// ---- launchers --------------------------------------------------------------

hipError_t launch_drift(const State& s, int n, double dt, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    k_drift<false><<<(n + 255) / 256, 256, 0, st>>>(s, s, n, dt);
    return hipGetLastError();
}

hipError_t launch_drift_to(const State& s, const State& d, int n, double dt, hipStream_t st)
{
    k_drift<true><<<(n + 255) / 256, 256, 0, st>>>(s, d, n, dt);
    return hipGetLastError();
}

hipError_t launch_copy_prev(const State& s, int n, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    k_copy_prev<<<(n + 255) / 256, 256, 0, st>>>(s, n);
    return hipGetLastError();
}

// Launch shapes of the ordered pair pass: balls per workgroup, pairs per lane and batch,
// wavefronts, rounds of 64 touching pairs before the turn, wavefronts per SIMD the registers are
// held to, pairs unrolled, scan.  All give the same results bit for bit.  The sizes at which each
// is the fastest are at ordered_default_shape; 8 has a few of the smallest (16 balls 6.74 us,
// shape 7 6.79); 2 and 6 have none of those measured (2 comes next after 5 at 1,100 to 1,500 balls
// and 3 at 1,800, 6 after 1 at 1,000) and stay because callers force shapes by these numbers.
#define SL_ORD_SHAPES(X) \
    X(0, 2, 2, 8, 2, 2, 2, true) \
    X(1, 4, 4, 8, 2, 2, 2, true) \
    X(2, 4, 4, 4, 1, 3, 2, true) \
    X(3, 4, 4, 4, 1, 3, 2, false) \
    X(4, 8, 4, 4, 1, 3, 2, false) \
    X(5, 2, 2, 4, 1, 3, 2, true) \
    X(6, 4, 2, 8, 2, 2, 2, true) \
    X(7, 2, 1, 8, 1, 2, 1, true) \
    X(8, 2, 1, 4, 1, 2, 1, true)

namespace {
#define SL_X(id, NB, CH, W, AD, WPE, UNR, SCAN) NB,
constexpr int ORD_BALLS[] = {SL_ORD_SHAPES(SL_X)};
#undef SL_X
constexpr int N_ORD_SHAPES = (int)(sizeof(ORD_BALLS) / sizeof(ORD_BALLS[0]));
}  // namespace

int ordered_shapes() { return N_ORD_SHAPES; }

int ordered_blocks(int n, int shape)
{
    const int nb = ORD_BALLS[(shape >= 0 && shape < N_ORD_SHAPES) ? shape : 0];
    return (n + nb - 1) / nb;
}

namespace {
hipError_t launch_ordered(const OrdState& os, const Phys& P, int n, int write, double* pe_ball,
                          unsigned long long* contacts, hipStream_t st, int shape)
{
    if (shape < 0 || shape >= N_ORD_SHAPES) shape = 0;
    const int nb = ordered_blocks(n, shape);
#define SL_X(id, NB, CH, W, AD, WPE, UNR, SCAN)                                                                     \
    case id:                                                                                                    \
        if (write)                                                                                              \
            k_pairs_ordered<NB, CH, W, AD, WPE, UNR, SCAN, true><<<nb, 64 * W, 0, st>>>(os, P, n, pe_ball, contacts);  \
        else                                                                                                    \
            k_pairs_ordered<NB, CH, W, AD, WPE, UNR, SCAN, false><<<nb, 64 * W, 0, st>>>(os, P, n, pe_ball, contacts); \
        break;
    switch (shape) {
        SL_ORD_SHAPES(SL_X)
    }
#undef SL_X
    return hipGetLastError();
}
}  // namespace

hipError_t launch_pairs_ordered(const State& s, const Phys& P, int n, int write, double* pe_ball,
                                unsigned long long* contacts, hipStream_t st, int shape)
{
    if (n <= 1) return hipSuccess;
    const OrdState os{s.f[0], s.f[0], nullptr, (long)(s.f[1] - s.f[0]), 0, nullptr};
    return launch_ordered(os, P, n, write, pe_ball, contacts, st, shape);
}

hipError_t launch_step_ordered(const double* konst, double* cur, double* nxt, long stride, const Phys& P, int n, int drift,
                               unsigned long long* contacts, int* nonfinite, hipStream_t st, int shape)
{
    const OrdState os{cur, konst, nxt, stride, drift, nonfinite};
    return launch_ordered(os, P, n, 0, nullptr, contacts, st, shape);
}

int kick_blocks(int n) { return (n + 255) / 256; }

hipError_t launch_kick(const State& s, int n, double dt, int write, int kick, double* e_part,
                       int* nonfinite, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    k_kick<<<kick_blocks(n), 256, 0, st>>>(s, n, dt, write, kick, e_part, nonfinite);
    return hipGetLastError();
}

}  // namespace sl
