// Device kernels of the fast path (included by sl_kernels_fast.hip).
//
//   k_tiles_*  SPLIT wavefronts per 64x64 tile (I, J) of a system's pair triangle,
//              I >= J, each sweeping 64/SPLIT of the tile's diagonals.  Lane l
//              holds ball i = 64 I + l in registers.  The 64 balls of block J are
//              staged in LDS twice (slots 0..63 and 64..127), so at sweep step s lane
//              l reads slot l + s -- ball j = (l + s) mod 64 -- at base + s*stride,
//              with no index arithmetic.  The reaction force on j is accumulated in
//              a register that travels with j: after every step the accumulators
//              rotate one lane down (DPP wave_rol:1), so lane l always holds the sum
//              of the j it meets next; no LDS atomics or cross-lane reductions.
//              A pair closer than S + h_min (touching, or in the band where the
//              reference clamps the vdW gap) contributes nothing to the sweep: it is
//              only recorded, as a bit of the partner masks of both balls.  The near
//              test's compare is already the wavefront's lane mask: a step with any
//              near lane stores that mask in LDS (a uniform branch, rarely taken), and
//              each lane's partner bits are rebuilt from the stored steps after the
//              sweep, so the sweep itself spends no vector instructions on them.  Each
//              tile writes its i-side and j-side force sums and partner masks once,
//              to slot J of the balls of block I and slot I of the balls of block J
//              (system-local block numbers), so every (ball, slot) that is read is written by
//              exactly one tile per step and nothing needs clearing (large systems: see
//              ROW_GROUP and the near marks).
//   k_ball     one workgroup per 64-ball block, eight or four wavefronts with lane
//              l working for ball l: the far-field partials of every eighth slot
//              (one slot class) are summed by one wavefront (Kahan-compensated in
//              the mixed mode), which counts the ball's partner-mask bits; the block
//              numbers its near pairs ball by ball and evaluates them with the
//              reference arithmetic, one per thread, in rounds of one entry per
//              thread; then each component of force and torque is finished by a
//              wavefront: the near results of each ball in entry order, acc and aacc, the
//              closing kick and the next step's drift (writing the
//              other state set).  A near pair is evaluated once for each of its two
//              balls, by the blocks that hold them.
// Every sum has a fixed order at a given tile split, so results are reproducible run
// to run; the k_ball shape does not change them.
#pragma once

#include "sl_fast_pair.hpp"
#include "sl_internal.hpp"
#include "sl_pair_ref.hpp"

#include <type_traits>

#pragma clang fp contract(off)

namespace sl {
namespace fastk {

constexpr int TB = FAST_TILE;
constexpr int NW = 4;                 // wavefronts per block
#ifndef SL_TILE_UNROLL
#define SL_TILE_UNROLL 2              // pairs of the tile sweep unrolled per wavefront
#endif
constexpr int NT = TB * NW;
constexpr int KB_C = 8;              // k_ball's slot classes K = c, c + KB_C, ...: they fix the order of every sum
constexpr int SLOTS_IN_FLIGHT = 10;  // slots per lane k_ball loads together: 40 loads
constexpr int KB_BATCH = SLOTS_IN_FLIGHT * KB_C;   // one batch for systems of up to 80 blocks

// Lane l receives the value held by lane (l + 1) mod 64 (DPP wave_rol:1).
__device__ __forceinline__ float rot1(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x134, 0xf, 0xf, false));
}
__device__ __forceinline__ double rot1(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)b, 0x134, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), 0x134, 0xf, 0xf, false);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
// Lane l receives the value held by lane (l + k) mod 64 (ds_bpermute).
__device__ __forceinline__ float rotk(float v, int k)
{
    const int src = ((int)(threadIdx.x % TB) + k) & (TB - 1);
    return __int_as_float(__builtin_amdgcn_ds_bpermute(src * 4, __float_as_int(v)));
}
__device__ __forceinline__ double rotk(double v, int k)
{
    const int src = ((int)(threadIdx.x % TB) + k) & (TB - 1);
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_ds_bpermute(src * 4, (int)b);
    const int hi = __builtin_amdgcn_ds_bpermute(src * 4, (int)(b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

__device__ __forceinline__ unsigned long long rotl64(unsigned long long x, int k)
{
    return k ? (x << k) | (x >> (64 - k)) : x;
}

// Systems of more than KB_BATCH blocks list their tiles in groups of NW of one row I, J = 4 g ..
// 4 g + 3 (the last group of a row is filled up with I = -1), and the binary64 sweep, where a
// workgroup takes several tiles, adds the i sides of a group's tiles before they go to memory:
// one partial instead of four (two, with two wavefronts a tile), in the slot of the group's
// first tile.  Per ball that leaves 5 of 8 partials to write and to read (the mixed sweep keeps
// them apart: binary32 sums depend on their order).  At 40,000 spheres the per-ball kernel went
// from 171 to 113 us (600 to 375 MB of partials) and the sweep from 1020 to 1005.  Smaller
// systems' partials are one batch of loads per ball and not what bounds them.
constexpr int ROW_GROUP = 1 << 30;

struct TileArgs {
    const double* px;
    const double* py;
    const double* pz;
    const double* R;
    FastAux aux;
    const Phys* sysP;       // per system
    const double4* bnd;     // per 64-ball block: bounding box of the centres (lo with max R, hi)
    const float4* xl;       // mixed: per ball, position relative to its block's box centre and R, in units of L0
    const double* gq_blk;   // per 64-ball block, the largest g/q of its balls (aux.g, aux.q): grav_share, both precisions
    int n_pad;
    int n_tiles;
    const int4* tiles;      // {I, J, system, first block of the system | ROW_GROUP}; I < 0: no tile
    float L0inv, L0inv2;    // mixed: 1 / L0 and 1 / L0^2 (scaled units)
    double Kf;              // mixed: force = Kf * (scaled binary32 factor) * (r / L0)
    double* part;           // [slot][xyz][n_pad]; the mixed mode stores binary32 sums, Kf left out,
                            // in the first half of the same buffer ([slot][xyz][n_pad] floats)
    unsigned long long* nbm;   // [slot][n_pad]: near-partner masks; with near, only where it is set
    unsigned char* near;    // per 64-ball block and slot (near_stride apart): the slot's masks have a bit
                            // set (NULL: every mask is written)
    int near_stride;
    double* pe_row;         // write steps: far-field energy of tile (I, J) at 64-ball block I's row
    int pe_stride;          // (pe_stride apart), slot J
    int* queue;             // k_tiles_q: next group per segment, workgroups done (all 0 between launches)
};

// Sum over the 64 lanes of a wavefront as a fixed tree (deterministic).
__device__ __forceinline__ double wave_sum(double v)
{
    for (int m = 1; m < TB; m <<= 1) v = v + __shfl_xor(v, m, TB);
    return v;
}

// Sums over lanes 0 .. l (DPP row shifts, then the rows' totals).
__device__ __forceinline__ int wave_iscan(int v)
{
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);   // row_shr:1, 2, 4, 8
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);   // row_bcast:15 to rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);   // row_bcast:31 to rows 2 and 3
    return v;
}

__device__ __forceinline__ int wave_isum(int v)
{
    for (int m = 1; m < TB; m <<= 1) v += __shfl_xor(v, m, TB);
    return v;
}

// Smallest and largest value of the valid lanes (every lane gets the result; +inf and -inf
// without any).  Quads, rows of 16 by DPP mirrors, then the four rows.
__device__ __forceinline__ void wave_minmax(double v, bool valid, double& lo, double& hi)
{
    const double inf = __builtin_huge_val();
    lo = valid ? v : inf;
    hi = valid ? v : -inf;
    auto mv = [](double d, auto ctrl) {
        const long long b = __double_as_longlong(d);
        const int l = __builtin_amdgcn_mov_dpp((int)b, decltype(ctrl)::value, 0xf, 0xf, false);
        const int h = __builtin_amdgcn_mov_dpp((int)(b >> 32), decltype(ctrl)::value, 0xf, 0xf, false);
        return __longlong_as_double((long long)(((unsigned long long)(unsigned)h << 32) | (unsigned)l));
    };
    auto step = [&](auto ctrl) {
        lo = fmin(lo, mv(lo, ctrl));
        hi = fmax(hi, mv(hi, ctrl));
    };
    step(std::integral_constant<int, 0xB1>{});    // quad_perm 1,0,3,2
    step(std::integral_constant<int, 0x4E>{});    // quad_perm 2,3,0,1
    step(std::integral_constant<int, 0x141>{});   // row_half_mirror
    step(std::integral_constant<int, 0x140>{});   // row_mirror
    auto lane = [](double d, int k) {
        const long long b = __double_as_longlong(d);
        const int l = __builtin_amdgcn_readlane((int)b, k), h = __builtin_amdgcn_readlane((int)(b >> 32), k);
        return __longlong_as_double((long long)(((unsigned long long)(unsigned)h << 32) | (unsigned)l));
    };
    const double l0 = fmin(lane(lo, 0), lane(lo, 16)), l1 = fmin(lane(lo, 32), lane(lo, 48));
    const double h0 = fmax(lane(hi, 0), lane(hi, 16)), h1 = fmax(lane(hi, 32), lane(hi, 48));
    lo = fmin(l0, l1);
    hi = fmax(h0, h1);
}

// Bounding box of the valid balls held one per lane (every lane gets the result):
// lo = (min x, min y, min z, max R), hi = (max x, max y, max z, 0).
__device__ __forceinline__ void wave_aabb(double x, double y, double z, double R, bool valid, double4& lo,
                                          double4& hi)
{
    double none, rm;
    wave_minmax(x, valid, lo.x, hi.x);
    wave_minmax(y, valid, lo.y, hi.y);
    wave_minmax(z, valid, lo.z, hi.z);
    wave_minmax(R, valid, none, rm);
    lo.w = fmax(rm, 0.0);
    hi.w = 0;
}

// A tile is far when the gap between its two blocks' bounding boxes exceeds the two
// largest radii plus h_min (with a 1e-9 relative margin): every pair in it is then
// farther apart than S + h_min by far more than the rounding of the per-pair test,
// so the sweep needs no near test.  Diagonal tiles always get the test.
__device__ __forceinline__ bool tile_is_far(const TileArgs& a, int I, int J, double h_min)
{
    if (I == J) return false;
    const double4 li = a.bnd[2 * I], ui = a.bnd[2 * I + 1], lj = a.bnd[2 * J], uj = a.bnd[2 * J + 1];
    const double gx = fmax(0.0, fmax(lj.x - ui.x, li.x - uj.x));
    const double gy = fmax(0.0, fmax(lj.y - ui.y, li.y - uj.y));
    const double gz = fmax(0.0, fmax(lj.z - ui.z, li.z - uj.z));
    const double lim = (li.w + lj.w + h_min) * (1 + 1e-9);
    return gx * gx + gy * gy + gz * gz > lim * lim;
}

// Largest share of gravity in the force of any pair of tile (I, J): g_i g_j / d^3 over
// q_i q_j / (s t)^2 is at most (g/q)_I (g/q)_J dmax^5, because s, t <= d^2 <= dmax^2 (dmax: the
// largest distance between the blocks' boxes).  NaN where a position is.  From the binary64
// weights: the mixed path's overflow at radii of 7e12 median ones, which made the share 0.
__device__ __forceinline__ double grav_share(const TileArgs& a, int I, int J)
{
    const double4 li = a.bnd[2 * I], ui = a.bnd[2 * I + 1], lj = a.bnd[2 * J], uj = a.bnd[2 * J + 1];
    const double ex = fmax(uj.x - li.x, ui.x - lj.x), ey = fmax(uj.y - li.y, ui.y - lj.y);
    const double ez = fmax(uj.z - li.z, ui.z - lj.z);
    const double d2m = ex * ex + ey * ey + ez * ez;
    return a.gq_blk[I] * a.gq_blk[J] * d2m * d2m * __builtin_sqrt(d2m);
}

// Largest y = 4 Ri Rj / (d^2 - (Ri - Rj)^2) of the pairs of tile (I, J), from the gap between the
// blocks' boxes and their largest radii; +inf where the boxes are not apart, NaN where a
// position is.
__device__ __forceinline__ double energy_reach(const TileArgs& a, int I, int J)
{
    const double4 li = a.bnd[2 * I], ui = a.bnd[2 * I + 1], lj = a.bnd[2 * J], uj = a.bnd[2 * J + 1];
    const double gx = fmax(0.0, fmax(lj.x - ui.x, li.x - uj.x));
    const double gy = fmax(0.0, fmax(lj.y - ui.y, li.y - uj.y));
    const double gz = fmax(0.0, fmax(lj.z - ui.z, li.z - uj.z));
    const double rm = fmax(li.w, lj.w), t = gx * gx + gy * gy + gz * gz - rm * rm;
    return t > 0 ? 4 * li.w * lj.w / t : __builtin_huge_val();
}

// Sweep range of part h of SPLIT: off-diagonal tiles sweep s = 0..63; diagonal
// tiles s = 1..32 (each unordered pair of the block once; s = 32 for the lower
// half of the lanes only).
template <int SPLIT>
__device__ __forceinline__ void sweep_range(bool diag, int h, int& s0, int& s1)
{
    if (!diag) {
        s0 = h * (TB / SPLIT);
        s1 = (h + 1) * (TB / SPLIT);
    } else {
        s0 = 1 + h * ((TB / 2) / SPLIT);
        s1 = 1 + (h + 1) * ((TB / 2) / SPLIT);
    }
}

__device__ __forceinline__ int4 fetch_tile(const TileArgs& a, int t, bool live)
{
    return live ? a.tiles[t] : make_int4(0, 0, 0, 0);
}

struct JRec64 {
    double x, y, z, R, q, g;
};
// The mixed path's record: the binary64 geometry, and the binary32 factors it uses as
// they are (radius in units of L0, cohesion and gravity weights), so no pair converts them.
struct JRecMix {
    double x, y, z, R;
    float Rs, q, g, pad;
};
static_assert(sizeof(JRecMix) == sizeof(JRec64), "both records share the LDS staging area");
// The mixed path's staging for a far tile (every pair farther apart than S + h_min): all
// binary32, ball j's block-local position shifted by the offset between the two blocks'
// reference points, so a pair's displacement is one binary32 subtraction per axis.  Three
// arrays rather than one record, so that lane l's reads at step s (slot l + s) are 16 or 4
// bytes apart from its neighbours': every LDS bank once per pass (a 32-byte record puts
// two lanes on each bank of a 16-byte read and eight on each of a 4-byte one).
struct JSoA32 {
    float4 p[2 * TB];   // x, y, z in units of L0 relative to block I's reference point; R / L0
    float q[2 * TB];    // cohesion weight
    float g[2 * TB];    // gravity weight
};
static_assert(sizeof(JSoA32) <= sizeof(JRec64) * 2 * TB, "all records share the LDS staging area");

// Reference point of a 64-ball block: the centre of its bounding box (lo, hi).
__device__ __forceinline__ double3 block_ref(double4 lo, double4 hi)
{
    return make_double3(0.5 * (lo.x + hi.x), 0.5 * (lo.y + hi.y), 0.5 * (lo.z + hi.z));
}

// The pair sweep of every tile: the far-field force of each pair, with the per-pair
// near test only in tiles the bounding-box test cannot rule out.  A near pair
// (closer than S + h_min) contributes nothing here; it is recorded as a bit of the
// partner masks of both balls, for k_ball.  SL_PREC_MIXED evaluates the factor in
// binary32, in units of L0 (median radius) and M0 (median mass), as one sum for vdW and
// gravity: f = Kf (q_i q_j / (s t)^2 + g_i g_j / d^3) with per-ball weights
// q = sqrt(Kv/Kf) (R/L0)^3, g = sqrt(Kg/Kf) m/M0, accumulated in binary32 per tile.  In
// far tiles of non-write steps the geometry is binary32 too (block-local coordinates);
// elsewhere it is binary64, rounded once the near test is done.  Each tile writes its i-side and
// j-side sums and masks once, to slot J of the balls of block I and slot I of the
// balls of block J, and its far-pair energy on write steps.
template <int PREC, bool WRITE, bool GRAV, int SPLIT>
__device__ __forceinline__ void tile_pass(const TileArgs& a, int tbase)
{
    constexpr int TPB = NW / SPLIT;
    constexpr size_t SJ_BYTES = sizeof(JRec64) * TPB * 2 * TB;
    constexpr size_t COMB_BYTES = sizeof(double) * NW * 6 * TB;
    __shared__ __attribute__((aligned(16))) unsigned char lds[SJ_BYTES > COMB_BYTES ? SJ_BYTES : COMB_BYTES];
    JRec64 (*sj)[2 * TB] = reinterpret_cast<JRec64 (*)[2 * TB]>(lds);
    double (*comb)[6][TB] = reinterpret_cast<double (*)[6][TB]>(lds);
    __shared__ double pe_w[NW];
    __shared__ unsigned long long im[TPB][TB], jm[TPB][TB];
    __shared__ unsigned long long bal[NW][TB];   // per wavefront: near lanes of step s

    // the wavefront index is uniform: in a scalar register, the tile and sweep indices
    // derived from it are too
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / TB), l = threadIdx.x % TB;
    const int tl = w / SPLIT, h = w % SPLIT;
    const int t = tbase + tl;
    int4 tt = fetch_tile(a, t, t < a.n_tiles);
    const bool live = t < a.n_tiles && tt.x >= 0;
    if (!live) tt = make_int4(0, 0, 0, 0);
    const int I = tt.x, J = tt.y, sys = tt.z, blk0 = tt.w & (ROW_GROUP - 1);
    const bool grouped = PREC == SL_PREC_FP64 && TPB > 1 && (tt.w & ROW_GROUP) != 0;
    const Phys& P = a.sysP[sys];
    const bool diag = I == J;
    const bool test = live && !tile_is_far(a, I, J, P.h_min);
    const int i = I * TB + l;
    const int j0 = J * TB + l;
    const double xi = a.px[i], yi = a.py[i], zi = a.pz[i], Ri = a.R[i];
    const double qi = PREC == SL_PREC_MIXED ? (double)a.aux.q32[i] : a.aux.q[i];
    const double gi = PREC == SL_PREC_MIXED ? (double)a.aux.g32[i] : a.aux.g[i];
    // mixed precision, far tile, no energies: the whole pair in binary32
    const bool f32 = PREC == SL_PREC_MIXED && !WRITE && live && !test;
    if (live && h == 0) {
        if (f32) {
            const double3 ci = block_ref(a.bnd[2 * I], a.bnd[2 * I + 1]);
            const double3 cj = block_ref(a.bnd[2 * J], a.bnd[2 * J + 1]);
            const double L0inv = (double)a.L0inv;
            const float4 xj = a.xl[j0];
            const float4 pj = make_float4(xj.x + (float)((cj.x - ci.x) * L0inv),
                                          xj.y + (float)((cj.y - ci.y) * L0inv),
                                          xj.z + (float)((cj.z - ci.z) * L0inv), xj.w);
            const float qj = a.aux.q32[j0], gj = a.aux.g32[j0];
            JSoA32* sm = reinterpret_cast<JSoA32*>(sj[tl]);
            sm->p[l] = pj;
            sm->p[l + TB] = pj;
            sm->q[l] = qj;
            sm->q[l + TB] = qj;
            sm->g[l] = gj;
            sm->g[l + TB] = gj;
        } else if constexpr (PREC == SL_PREC_MIXED) {
            JRecMix r;
            r.x = a.px[j0];
            r.y = a.py[j0];
            r.z = a.pz[j0];
            r.R = a.R[j0];
            r.Rs = (float)a.R[j0] * a.L0inv;
            r.q = a.aux.q32[j0];
            r.g = a.aux.g32[j0];
            r.pad = 0.f;
            JRecMix* sm = reinterpret_cast<JRecMix*>(sj[tl]);
            sm[l] = r;
            sm[l + TB] = r;
        } else {
            JRec64 r;
            r.x = a.px[j0];
            r.y = a.py[j0];
            r.z = a.pz[j0];
            r.R = a.R[j0];
            r.q = a.aux.q[j0];
            r.g = a.aux.g[j0];
            sj[tl][l] = r;
            sj[tl][l + TB] = r;
        }
        im[tl][l] = 0;
        jm[tl][l] = 0;
    }
    __syncthreads();

    double ax = 0, ay = 0, az = 0, bx = 0, by = 0, bz = 0, pe = 0, pg = 0;
    unsigned long long any = 0;         // bit s: some lane met a near pair at step s
    if (live) {
        const JRec64* rec = &sj[tl][l];
        const double Ri4 = 4 * Ri;
        const double h_min = P.h_min;
        const double hmin2 = h_min * h_min, two_hmin = 2 * h_min;
        const bool efar = WRITE && !test && energy_reach(a, I, J) <= 0x1p-5;
        int s0, s1;
        sweep_range<SPLIT>(diag, h, s0, s1);
        if (PREC == SL_PREC_MIXED && f32) {
            // far tile: displacement, distance, the vdW and gravity factor and the sums
            // all in binary32, in units of L0 and M0 (no near test: the box test cleared
            // every pair)
            const float4 xi4 = a.xl[i];
            const float qif = a.aux.q32[i], gif = a.aux.g32[i];
            const float r4i = 4.0f * xi4.w;
            float fax = 0.f, fay = 0.f, faz = 0.f, fbx = 0.f, fby = 0.f, fbz = 0.f;
            const JSoA32* soa = reinterpret_cast<const JSoA32*>(sj[tl]);
            const float4* rp32 = soa->p + l;
            const float* rq32 = soa->q + l;
            const float* rg32 = soa->g + l;
            // Gravity is left out of a tile whose every pair has it below 2^-27 of the vdW
            // term: added by the FMA it would be under half an ulp of the factor, so leaving
            // it out changes no bit.
            const bool grav = GRAV && !(grav_share(a, I, J) < 0x1p-27);
            auto pair32 = [&](int s, auto gv) {
                const float4 rp = rp32[s];
                const float dx = rp.x - xi4.x, dy = rp.y - xi4.y, dz = rp.z - xi4.z;
                const float d2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
                const float S = xi4.w + rp.w;
                const float sv = __builtin_fmaf(-S, S, d2);
                const float tv = __builtin_fmaf(r4i, rp.w, sv);
                const float st = sv * tv;
                float f = (qif * rq32[s]) * __builtin_amdgcn_rcpf(st * st);
                if constexpr (decltype(gv)::value) {
                    const float rq = __builtin_amdgcn_rsqf(d2);
                    f = __builtin_fmaf(gif * rg32[s], rq * rq * rq, f);
                }
                fax = __builtin_fmaf(f, dx, fax);
                fay = __builtin_fmaf(f, dy, fay);
                faz = __builtin_fmaf(f, dz, faz);
                fbx = rot1(__builtin_fmaf(-f, dx, fbx));
                fby = rot1(__builtin_fmaf(-f, dy, fby));
                fbz = rot1(__builtin_fmaf(-f, dz, fbz));
            };
            {
                constexpr int NS = TB / SPLIT;
                if (GRAV && grav) {
#pragma unroll SL_TILE_UNROLL
                    for (int k = 0; k < NS; k++) pair32(s0 + k, std::true_type{});
                } else {
#pragma unroll SL_TILE_UNROLL
                    for (int k = 0; k < NS; k++) pair32(s0 + k, std::false_type{});
                }
            }
            const int back = (TB - (s1 & (TB - 1))) & (TB - 1);
            if (back) {
                fbx = rotk(fbx, back);
                fby = rotk(fby, back);
                fbz = rotk(fbz, back);
            }
            // binary32 sums, exact in binary64 (Kf is applied in k_ball)
            ax = fax; ay = fay; az = faz;
            bx = fbx; by = fby; bz = fbz;
        } else if constexpr (PREC == SL_PREC_MIXED) {
            const float qif = (float)qi, gif = (float)gi, L0inv2 = a.L0inv2, L0inv = a.L0inv;
            const float r4i = 4.0f * (float)Ri * L0inv;
            float fax = 0.f, fay = 0.f, faz = 0.f, fbx = 0.f, fby = 0.f, fbz = 0.f;
            const JRecMix* recm = reinterpret_cast<const JRecMix*>(sj[tl]) + l;
            auto pair = [&](int s, bool act, auto ntest, auto efar) {
                const JRecMix& r = recm[s];
                const double dx = r.x - xi, dy = r.y - yi, dz = r.z - zi;
                const double d2 = __builtin_fma(dz, dz, __builtin_fma(dy, dy, dx * dx));
                const double S = Ri + r.R;
                const double sv = __builtin_fma(-S, S, d2);
                const float s32 = (float)sv * L0inv2;
                const float t32 = __builtin_fmaf(r4i, r.Rs, s32);
                const float st = s32 * t32;
                float f = (qif * r.q) * __builtin_amdgcn_rcpf(st * st);
                if (GRAV) {
                    const float rq = __builtin_amdgcn_rsqf((float)d2 * L0inv2);
                    f = __builtin_fmaf(gif * r.g, rq * rq * rq, f);
                }
                bool use = true;
                if constexpr (decltype(ntest)::value) {
                    const bool near = sv < __builtin_fma(S, two_hmin, hmin2);
                    use = act && !near;
                    f = use ? f : 0.f;
                    const unsigned long long b = __ballot(act && near);
                    if (b) {
                        if (l == 0) bal[w][s] = b;
                        any |= 1ull << s;
                    }
                }
                // the unit scale on the factor once, not on each displacement
                f = f * L0inv;
                const float dxf = (float)dx, dyf = (float)dy, dzf = (float)dz;
                fax = __builtin_fmaf(f, dxf, fax);
                fay = __builtin_fmaf(f, dyf, fay);
                faz = __builtin_fmaf(f, dzf, faz);
                fbx = rot1(__builtin_fmaf(-f, dxf, fbx));
                fby = rot1(__builtin_fmaf(-f, dyf, fby));
                fbz = rot1(__builtin_fmaf(-f, dzf, fbz));
                if (WRITE) {
                    const double tv = __builtin_fma(Ri4, r.R, sv);
                    const double u = far_energy<decltype(efar)::value>(Ri, r.R, sv, tv, use);
                    pe = use ? pe + u : pe;
                    if (GRAV) {
                        const double gg = a.aux.g[i] * a.aux.g[J * TB + ((l + s) & (TB - 1))];
                        pg = use ? __builtin_fma(gg, rsq_f64(d2), pg) : pg;
                    }
                }
            };
            auto sweep = [&](auto ntest, auto efar) {
                if (!diag) {
                    constexpr int NS = TB / SPLIT;
                    if constexpr (WRITE) {
                        for (int k = 0; k < NS; k++) pair(s0 + k, true, ntest, efar);
                    } else {
#pragma unroll SL_TILE_UNROLL
                        for (int k = 0; k < NS; k++) pair(s0 + k, true, ntest, efar);
                    }
                } else {
                    for (int s = s0; s < s1 - 1; s++) pair(s, true, ntest, efar);
                    pair(s1 - 1, s1 - 1 < TB / 2 || l < TB / 2, ntest, efar);
                }
            };
            if (test)
                sweep(std::true_type{}, std::false_type{});
            else if (!efar)
                sweep(std::false_type{}, std::false_type{});
            else if constexpr (WRITE)
                sweep(std::false_type{}, std::true_type{});
            const int back = (TB - (s1 & (TB - 1))) & (TB - 1);
            if (back) {
                fbx = rotk(fbx, back);
                fby = rotk(fby, back);
                fbz = rotk(fbz, back);
            }
            // binary32 sums, exact in binary64 (Kf is applied in k_ball)
            ax = fax; ay = fay; az = faz;
            bx = fbx; by = fby; bz = fbz;
        } else {
            // Where gravity is below 2^-31 of the vdW term in every pair of the tile, the
            // hardware's reciprocal square root serves as it is: its cube's 2^-22.8 is then
            // less than half an ulp of the factor (the Newton step's cube has 2^-44).  Four of the
            // pair's 37 instructions; nearly all tiles of an aggregate of dust (at 5,000
            // spheres of 1e-5 cm the largest share is 2^-33, at 40,000 2^-29).  The sweep at
            // 40,000 went from 1141 to 1020 us, at 5,000 from 28.6 to 27.5, of 96 uneven
            // systems of up to 4,500 from 225 to 207.
            auto pair = [&](int s, bool act, auto ntest, auto raw, auto efar) {
                const JRec64& r = rec[s];
                const double dx = r.x - xi, dy = r.y - yi, dz = r.z - zi;
                const double Rj = r.R;
                const double d2 = __builtin_fma(dz, dz, __builtin_fma(dy, dy, dx * dx));
                const double S = Ri + Rj;
                const double sv = __builtin_fma(-S, S, d2);      // d^2 - S^2
                const double tv = __builtin_fma(Ri4, Rj, sv);    // d^2 - (Ri - Rj)^2
                const double st = sv * tv;
                double f = (qi * r.q) * rcp_f64(st * st);
                double rinv = 0;
                if (GRAV) {
                    rinv = decltype(raw)::value ? __builtin_amdgcn_rsq(d2) : rsq_f64(d2);
                    f = __builtin_fma(gi * r.g, rinv * rinv * rinv, f);
                }
                bool use = true;
                if constexpr (decltype(ntest)::value) {
                    const bool near = sv < __builtin_fma(S, two_hmin, hmin2);   // (S + h_min)^2 - S^2
                    use = act && !near;
                    f = use ? f : 0.0;
                    const unsigned long long b = __ballot(act && near);
                    if (b) {
                        if (l == 0) bal[w][s] = b;
                        any |= 1ull << s;
                    }
                }
                ax = __builtin_fma(f, dx, ax);
                ay = __builtin_fma(f, dy, ay);
                az = __builtin_fma(f, dz, az);
                bx = rot1(__builtin_fma(-f, dx, bx));
                by = rot1(__builtin_fma(-f, dy, by));
                bz = rot1(__builtin_fma(-f, dz, bz));
                if (WRITE) {
                    const double u = far_energy<decltype(efar)::value>(Ri, Rj, sv, tv, use);
                    pe = use ? pe + u : pe;
                    // (gravity's share of the energy is at most 6 times that of the force)
                    if (GRAV) pg = use ? __builtin_fma(gi * r.g, rinv, pg) : pg;
                }
            };
            auto sweep = [&](auto ntest, auto raw, auto efar) {
                if (!diag) {
                    constexpr int NS = TB / SPLIT;
                    if constexpr (WRITE) {
                        for (int k = 0; k < NS; k++) pair(s0 + k, true, ntest, raw, efar);
                    } else {
#pragma unroll SL_TILE_UNROLL
                        for (int k = 0; k < NS; k++) pair(s0 + k, true, ntest, raw, efar);
                    }
                } else {
                    for (int s = s0; s < s1 - 1; s++) pair(s, true, ntest, raw, efar);
                    pair(s1 - 1, s1 - 1 < TB / 2 || l < TB / 2, ntest, raw, efar);
                }
            };
            const bool raw = GRAV && grav_share(a, I, J) < 0x1p-31;
            auto go = [&](auto rw) {
                if (test)
                    sweep(std::true_type{}, rw, std::false_type{});
                else if (!efar)
                    sweep(std::false_type{}, rw, std::false_type{});
                else if constexpr (WRITE)
                    sweep(std::false_type{}, rw, std::true_type{});
            };
            if (raw)
                go(std::true_type{});
            else
                go(std::false_type{});
            const int back = (TB - (s1 & (TB - 1))) & (TB - 1);
            if (back) {
                bx = rotk(bx, back);
                by = rotk(by, back);
                bz = rotk(bz, back);
            }
        }
        // this lane's near steps, from the wavefront's recorded steps
        unsigned long long nmask = 0;
        for (unsigned long long z = any; z; z &= z - 1) {
            const int s = __ffsll((long long)z) - 1;
            if ((bal[w][s] >> l) & 1ull) nmask |= 1ull << s;
        }
        if (nmask) {
            atomicOr(&im[tl][l], rotl64(nmask, l));
            unsigned long long m = nmask;
            while (m) {
                const int s = __ffsll((long long)m) - 1;
                m &= m - 1;
                atomicOr(&jm[tl][(l + s) & (TB - 1)], 1ull << l);
            }
        }
        if (WRITE) {
            const double ws = wave_sum(-P.Ha / 6 * pe - pg);
            if (l == 0) pe_w[w] = ws;
        }
    }
    __syncthreads();
    if (live) {
        comb[w][0][l] = ax;
        comb[w][1][l] = ay;
        comb[w][2][l] = az;
        comb[w][3][l] = bx;
        comb[w][4][l] = by;
        comb[w][5][l] = bz;
    }
    __syncthreads();
    if (grouped && h == 0 && live && tl == 0) {
        // the i sides of the group's tiles, J to the diagonal (whose j side is on the same balls)
        const int in_group = min(TPB, I - J + 1);
        for (int k = 0; k < 3; k++) {
            double acc = 0;
            for (int g = 0; g < in_group; g++) {
                for (int q = 0; q < SPLIT; q++) acc = acc + comb[g * SPLIT + q][k][l];
                if (J + g == I)
                    for (int q = 0; q < SPLIT; q++) acc = acc + comb[g * SPLIT + q][k + 3][l];
            }
            a.part[((size_t)(J - blk0) * 3 + k) * a.n_pad + i] = acc;
        }
    }
    if (!(live && h == 0)) return;
    const int w0 = tl * SPLIT;
    const size_t np = (size_t)a.n_pad;
    const size_t si = (size_t)(J - blk0), sj_ = (size_t)(I - blk0);
    const unsigned long long mi = im[tl][l], mj = jm[tl][l];
    // The mixed mode's partials are binary32: the wavefronts' sums (binary32 values, held
    // exactly in comb) are added in binary32 and stored in the first half of the buffer.
    using PT = std::conditional_t<PREC == SL_PREC_MIXED, float, double>;
    PT v[6];
    for (int k = 0; k < 6; k++) {
        PT acc = (PT)comb[w0][k][l];
        for (int q = 1; q < SPLIT; q++) acc = acc + (PT)comb[w0 + q][k][l];
        v[k] = acc;
    }
    PT* part = reinterpret_cast<PT*>(a.part);
    if (diag) {
        // the i side and the j side of the diagonal tile land on the same balls
        if (!grouped) {
            part[(si * 3 + 0) * np + i] = v[0] + v[3];
            part[(si * 3 + 1) * np + i] = v[1] + v[4];
            part[(si * 3 + 2) * np + i] = v[2] + v[5];
        }
        const bool near = !a.near || __any((mi | mj) != 0);
        if (near) a.nbm[si * np + i] = mi | mj;
        if (a.near && l == 0) a.near[(size_t)I * a.near_stride + si] = near;
    } else {
        if (!grouped) {
            part[(si * 3 + 0) * np + i] = v[0];
            part[(si * 3 + 1) * np + i] = v[1];
            part[(si * 3 + 2) * np + i] = v[2];
        }
        part[(sj_ * 3 + 0) * np + j0] = v[3];
        part[(sj_ * 3 + 1) * np + j0] = v[4];
        part[(sj_ * 3 + 2) * np + j0] = v[5];
        const bool near = !a.near || __any(mi != 0);   // a pair sets a bit on both sides
        if (near) {
            a.nbm[si * np + i] = mi;
            a.nbm[sj_ * np + j0] = mj;
        }
        if (a.near && l == 0) {
            a.near[(size_t)I * a.near_stride + si] = near;
            a.near[(size_t)J * a.near_stride + sj_] = near;
        }
    }
    if (WRITE && l == 0) {
        double pt = pe_w[w0];
        for (int q = 1; q < SPLIT; q++) pt = pt + pe_w[w0 + q];
        a.pe_row[(size_t)I * a.pe_stride + si] = pt;
    }
}

// One launch, one workgroup per TPB tiles of the list.
template <int PREC, bool WRITE, bool GRAV, int SPLIT>
__global__ __launch_bounds__(NT) void k_tiles(TileArgs a)
{
    tile_pass<PREC, WRITE, GRAV, SPLIT>(a, blockIdx.x * (NW / SPLIT));
}

// The same tiles from a work queue: as many workgroups as fit on the device at once, each
// taking the next group of TPB tiles until none is left.  The list is cut into QSEG
// segments with a counter each, QPAD ints apart (device-scope atomics on one cache line
// serialise, some 10-30 ns apiece); workgroup b starts on segment b mod QSEG and, when
// that is empty, takes from the others in turn.  Every tile runs the same code as in
// k_tiles, so the results are the same bits.  queue[QPAD s] is segment s's next group,
// queue[QPAD QSEG] counts the workgroups done; the last one rewinds them all for the next
// launch, after every workgroup has taken its last item.
constexpr int QSEG = 8;
constexpr int QPAD = 64;   // 256 bytes between counters
template <int PREC, bool WRITE, bool GRAV, int SPLIT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(WRITE ? 1 : 6))) void k_tiles_q(TileArgs a)
{
    constexpr int TPB = NW / SPLIT;
    __shared__ int next;
    const int groups = (a.n_tiles + TPB - 1) / TPB;
    const int seg0 = blockIdx.x % QSEG;
    for (int k = 0; k < QSEG; k++) {
        const int seg = (seg0 + k) % QSEG;
        const int g0 = (int)((long long)groups * seg / QSEG), g1 = (int)((long long)groups * (seg + 1) / QSEG);
        for (;;) {
            if (threadIdx.x == 0) next = g0 + atomicAdd(a.queue + QPAD * seg, 1);
            __syncthreads();
            const int g = __builtin_amdgcn_readfirstlane(next);   // uniform: scalar registers
            __syncthreads();   // every thread has read `next` before it is written again
            if (g >= g1) break;
            tile_pass<PREC, WRITE, GRAV, SPLIT>(a, g * TPB);
            __syncthreads();   // the pass's LDS is reused by the next item
        }
    }
    if (threadIdx.x == 0) {
        __threadfence();
        if (atomicAdd(a.queue + QPAD * QSEG, 1) == (int)gridDim.x - 1)
            for (int q = 0; q <= QSEG; q++) atomicExch(a.queue + QPAD * q, 0);
    }
}

// A near pair's dynamic state for pair_ref.
struct NearState {
    const TouchState& ts;
    __device__ D3 vA() const { return ts.vA; }
    __device__ D3 vB() const { return ts.vB; }
    __device__ D3 wA() const { return ts.wA; }
    __device__ D3 wB() const { return ts.wB; }
    __device__ double old_dist() const { return norm(ts.q); }
};

// The engine's state: dynamic field f of ball b at cur[f np + b], the fields both sets
// share (radius, mass, moment of inertia) at konst.
struct EngineState {
    const double* cur;
    const double* konst;
    size_t np;
    __device__ double at(int f, int b) const { return cur[f * np + b]; }
    __device__ D3 at3(int f, int b) const { return d3(at(f, b), at(f + 1, b), at(f + 2, b)); }
    __device__ double c(int f, int b) const { return konst[f * np + b]; }
};

// The near pair of ball b and partner p in the reference's orientation: A is the ball with the
// larger index in the caller's numbering (the friction terms are not symmetric in A and B).
// Everything is loaded at once, before the orientation and whether the pair touches are known
// (in an aggregate nearly every near pair touches): one trip to memory where there were three.
struct NearPair {
    PairIn in;
    TouchState ts;
    bool is_a;    // b is A
};
__device__ __forceinline__ NearPair near_load(const EngineState& c, const int* perm, int b, int p)
{
    const int cb = perm[b], cp = perm[p];
    const D3 xb = c.at3(PX, b), xp = c.at3(PX, p), vb = c.at3(VX, b), vp = c.at3(VX, p);
    const D3 wb = c.at3(WX, b), wp = c.at3(WX, p), qb = c.at3(QX, b), qp = c.at3(QX, p);
    const double Rb = c.c(RAD, b), Rp = c.c(RAD, p), mb = c.c(MASS, b), mp = c.c(MASS, p);
    const bool is_a = cb > cp;
    auto sel = [is_a](D3 x, D3 y) { return d3(is_a ? x.x : y.x, is_a ? x.y : y.y, is_a ? x.z : y.z); };
    return NearPair{{sel(xb, xp), sel(xp, xb), is_a ? Rb : Rp, is_a ? Rp : Rb, is_a ? mb : mp, is_a ? mp : mb},
                    {sel(vb, vp), sel(vp, vb), sel(wb, wp), sel(wp, wb), sel(qp, qb) - sel(qb, qp)},
                    is_a};
}

// Its evaluation in the reference's arithmetic: force and torque on b to f[0 .. 5], fs apart;
// the pair's energy when b is A to pe; returns bit 0: touching and b is A, bit 1: b is A.
template <bool WRITE>
__device__ __forceinline__ int near_eval(const NearPair& z, const Phys& P, double* f, int fs, double& pe)
{
    const PairIn& in = z.in;
    const D3 r = in.pB - in.pA;
    const double d2 = dot(r, r);
    PairOut o;
    bool done = FarRange::params(P) && FarRange::ball(in.RA, in.mA) && FarRange::ball(in.RB, in.mB) && FarRange::distance2(d2);
    if (done) {
        double dist, y;
        sqrt_rcp(d2, dist, y);
        done = (in.RA + in.RB) - dist > 0 && touch_pair_ref(P, WRITE, in, z.ts, o);
    }
    if (!done) pair_ref(P, WRITE, in, NearState{z.ts}, o);
    const D3 F = z.is_a ? o.F : -o.F;
    const D3 T = z.is_a ? o.tA : o.tB;
    f[0] = F.x; f[fs] = F.y; f[2 * fs] = F.z;
    f[3 * fs] = T.x; f[4 * fs] = T.y; f[5 * fs] = T.z;
    pe = z.is_a ? o.pe : 0.0;
    return z.is_a ? o.contact | 2 : 0;
}

struct BallArgs {
    const double* cur;  // state sets, as in EngineState
    double* nxt;
    const double* konst;
    const Phys* sysP;
    const int4* blk_info;   // per 64-ball block: {first slot, balls, blocks of its system, system}
    int n_pad;
    const double* part;     // [slot][xyz][n_pad]; mixed: binary32, to be scaled by Kf
    int group;              // binary64, systems of more than KB_BATCH blocks: tiles to an i-side partial
    double Kf;
    const unsigned long long* nbm;   // near-partner masks; NEARF: of the slots that near marks
    const unsigned char* near;
    int near_stride;
    const int* perm;    // engine slot -> the caller's ball index (fixes near-pair orientation)
    int kick, drift_next;
    double4* bnd;       // per 64-ball block: bounding box of the drifted positions (lo, hi)
    float4* xl;         // per ball: drifted position relative to its block's box centre, R (units of L0)
    double L0inv;
    const double* pe_row;   // write steps: far-field energies of the block's tiles, as in TileArgs
    int pe_stride;
    double* e_blk;      // FAST_E_STRIDE doubles per 64-ball block (write steps)
    unsigned long long* blk_ctr;   // per 64-ball block: running sums of touching and near pairs
    int* flags;         // [1]: a non-finite state appeared
};

// One coordinate of a ball's block-local binary32 position, in a block whose bounding box is
// [lo, hi] there; padding lanes get far, distinct, finite places (their weights are 0, so they
// add nothing).
__device__ __forceinline__ float local_coord(double x, bool valid, double lo, double hi, double L0inv, int l)
{
    return valid ? (float)((x - 0.5 * (lo + hi)) * L0inv) : 1e6f + 2048.f * (float)l;
}

constexpr int BPB = TB;              // balls per k_ball block
// k_ball workgroups have 8 wavefronts (one slot class each: the fewest dependent loads
// per wavefront, for a lone system of few blocks) or 4 (two classes each, at most 170 VGPRs
// and 53 KB of LDS: three workgroups share a CU, for launches of more blocks than CUs).
// The results are the same bit for bit.
constexpr int kb_threads(int nwv) { return nwv * TB; }

// One 64-ball block per workgroup; lane l of every wavefront works for ball l.  The
// slots of the block fall into KB_C classes, K = c, c + KB_C, ...; wavefront w takes the
// classes c = w, w + NWV, ...
//
// 1. For each of its classes a wavefront sums the far-field partials in slot order
//    (reads of 64 consecutive doubles; in the mixed mode binary32 sums scaled by Kf
//    and added with Kahan compensation), counts
//    the near-partner bits and keeps the first MC nonzero partner masks of each ball
//    in LDS (more than that: they are read again).
// 2. The block's near entries are numbered ball by ball (then by class, slot and bit; every
//    wavefront makes the same scan of the counts), and all threads evaluate them, one round
//    of NWV * 64 at a time, with the reference arithmetic and orientation.  Each near pair is
//    so evaluated once from each of its balls, identically, and no sum needs an atomic.
// 3. The step is finished component by component: wavefront q adds component q (force, then
//    torque) of its balls' near results in entry order and of the class sums in a fixed order
//    and carries that axis through kick, drift and bounding box; component 6 is the pair
//    counts.  (Wavefront 0 alone took 5,200 cycles for what is now about 2,000.)
//
// Bound by latency: a chain of four trips to memory (the block's table, the partials, the near
// pairs' state, each a kernel's worth of L2 misses) and of the touching pair's arithmetic,
// with one workgroup on a CU.  Finishing by component, both balls' state loaded at once, the
// pair's short divisions (touch_pair_ref), scans by DPP and the sums' loads kept in flight
// behind the pairs took it from 12.6 to 9.4 us at 1,000 spheres, from 13.2 to 11.2 at 5,000
// (mixed 12.6 to 10.8), from 40 to 32 for 512 systems of 33 to 550 and from 56 to 49 for 96 of
// 200 to 4,500.
//
// Write steps: the far-field energies of the block's tiles are added here, lane l those of slots
// l, l + 64, ... and then the lanes as a tree, so that a step brings ten values per block to
// the host (at 40,000 spheres, 195,625 tiles' energies copied and added there took 1 ms).
//
// NEARF, for systems of more than KB_BATCH slots: the masks of slots without near pairs, nine
// in ten of a large system's, are neither written nor read (a quarter of what there was to
// read at 40,000 spheres: 201 -> 170 us).  Smaller systems load one batch of masks unseen: finding
// out which first cost 0.4 us of 11 at 79 slots and 5 of 49 in the four-wavefront shape.
template <bool COMP, bool WRITE, int NWV, bool NEARF>
__global__ __launch_bounds__(kb_threads(NWV)) void k_ball(BallArgs a)
{
    static_assert(NWV == 8 || (NWV == 4 && !NEARF), "8 or 4 wavefronts; NEARF: one class each");
    constexpr int KB_W = NWV;                 // wavefronts
    constexpr int KB_T = kb_threads(NWV);     // threads, and near entries per round
    constexpr int KB_MC = NWV == 8 ? 4 : 2;   // partner masks kept per (class, ball)
    constexpr int NQ = 7;                     // components: force, torque, pair counts
    constexpr int QW = 8 / NWV;               // of these a wavefront has w, w + NWV
    // One class a wavefront: its sums' loads stay in flight behind the near pairs' evaluation
    constexpr bool SUMS_LATE = NWV == KB_C;
    __shared__ double sf[KB_C][3][TB];       // far-field force sums per class
    __shared__ int s_cnt[KB_C][TB];          // near entries per (class, ball)
    __shared__ int s_nm[KB_C][TB];           // slots of (class, ball) with near partners
    __shared__ int ent[KB_T];                // entries of the current round
    __shared__ double res[6][KB_T];          // their forces and torques
    __shared__ double res_pe[WRITE ? KB_T : 1];
    __shared__ unsigned char res_fl[KB_T];
    __shared__ unsigned long long s_mk[KB_C][KB_MC][TB];   // nonzero partner masks ...
    __shared__ int s_mks[KB_C][KB_MC][TB];                  // ... and their slots
    __shared__ double fin[WRITE ? 9 : 1][TB];               // v, w, position (write steps)
    // the wavefront index is uniform: in a scalar register, the slot indices derived from
    // it are too
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / TB), l = threadIdx.x % TB;
    const int i = blockIdx.x * TB + l;
    // NEARF: slots of a class that have near pairs, a byte each: 60 of them (six batches of
    // SLOTS_IN_FLIGHT) a load, the first while the block's table is on its way
    auto near_bytes = [&](int K0) {
        const int K = K0 + KB_C * l;
        return NEARF && l < 60 && K < a.near_stride ? (int)a.near[(size_t)blockIdx.x * a.near_stride + K] : 0;
    };
    const int near0 = near_bytes(w);
    const int4 bi = a.blk_info[blockIdx.x];
    const int off = bi.x, nb = bi.z;
    const bool valid = i - off < bi.y;
    const int ic = valid ? i : off;
    const Phys P = a.sysP[bi.w];
    const size_t np = (size_t)a.n_pad;
    const EngineState c{a.cur, a.konst, np};
    // far-field partials: binary32 in the mixed mode (the force is Kf times the stored sum)
    using PT = std::conditional_t<COMP, float, double>;
    const double Kf = a.Kf;

    // what this wavefront's components need of the balls' own state goes out first
    double x0[QW], h0[QW], inr[QW], Rb = 0;
    unsigned long long ctr0 = 0, ctr1 = 0;
    double far_pe = 0;   // lane l: slots l, l + 64, ... of the block's row of far-field energies
#pragma unroll
    for (int u = 0; u < QW; u++) {
        const int q = w + u * NWV;
        x0[u] = h0[u] = 0;
        inr[u] = 1;
        if (q < 3) {
            x0[u] = c.at(PX + q, ic);
            h0[u] = c.at(HX + q, ic);
            inr[u] = c.c(MASS, ic);
        } else if (q < 6) {
            h0[u] = c.at(GX + q - 3, ic);
            inr[u] = c.c(MOI, ic);
            if (q == 3) Rb = c.c(RAD, ic);
        } else if (q == 6) {
            if (l == 0) {
                ctr0 = a.blk_ctr[2 * blockIdx.x];
                ctr1 = a.blk_ctr[2 * blockIdx.x + 1];
            }
            if (WRITE)
                for (int J = l; J <= (int)blockIdx.x - off / TB; J += TB) far_pe = far_pe + a.pe_row[(size_t)blockIdx.x * a.pe_stride + J];
        }
    }

    // slots K0, K0 + KB_C, ... of a class: SLOTS_IN_FLIGHT loaded together (4 for small systems)
    const bool wide = nb > 4 * KB_C;
    auto slot = [&](int K0, int u) { return K0 + u * KB_C < nb ? K0 + u * KB_C : nb - 1; };
    // the block's sums, one after another: those of the groups up to the diagonal, then of the rows below
    const int grp = !COMP && nb > KB_BATCH ? a.group : 1;
    const int row = blockIdx.x - off / TB, ng = row / grp + 1, nsum = ng + nb - 1 - row;
    auto each_slot = [&](auto f) {
#pragma unroll
        for (int u = 0; u < 4; u++) f(u);
        if (wide) {
#pragma unroll
            for (int u = 4; u < SLOTS_IN_FLIGHT; u++) f(u);
        }
    };
    // masks of the batch at K0 (NEARF: bit u of near, its slot u has any)
    auto load_masks = [&](int K0, unsigned long long near, unsigned long long* mk) {
        each_slot([&](int u) {
            if constexpr (NEARF) {
                mk[u] = 0;
                if ((near >> u) & 1) mk[u] = a.nbm[(size_t)(K0 + u * KB_C) * np + ic];
            } else {
                mk[u] = a.nbm[(size_t)slot(K0, u) * np + ic];
            }
        });
    };
    auto near_slots = [&](int K0, int byte) { return __ballot(byte != 0 && K0 + KB_C * l < nb); };
    auto load_sums = [&](int K0, PT (*q)[3]) {
        each_slot([&](int u) {
            const int e = min(K0 + u * KB_C, nsum - 1), K = e < ng ? e * grp : row + 1 + e - ng;
            const PT* pp = reinterpret_cast<const PT*>(a.part) + (size_t)K * 3 * np + ic;
            q[u][0] = pp[0];
            q[u][1] = pp[np];
            q[u][2] = pp[2 * np];
        });
    };
    struct Near {
        int cn, nm;   // near entries of this (class, ball), slots that have any
    };
    auto count = [&](int cl, int K0, const unsigned long long* mk, Near& t) {
        each_slot([&](int u) {
            const unsigned long long m = valid && K0 + u * KB_C < nb ? mk[u] : 0ull;
            t.cn += __popcll(m);
            if (m) {
                if (t.nm < KB_MC) {
                    s_mk[cl][t.nm][l] = m;
                    s_mks[cl][t.nm][l] = K0 + u * KB_C;
                }
                t.nm++;
            }
        });
    };
    struct Sum {
        double f[3], c[3];
    };
    auto add = [&](int K0, PT (*q)[3], Sum& t) {
        each_slot([&](int u) {
            if (K0 + u * KB_C >= nsum) return;
#pragma unroll
            for (int x = 0; x < 3; x++) {
                if (COMP) {
                    const double y = Kf * (double)q[u][x] - t.c[x], z = t.f[x] + y;
                    t.c[x] = (z - t.f[x]) - y;
                    t.f[x] = z;
                } else {
                    t.f[x] = t.f[x] + q[u][x];
                }
            }
        });
    };
    PT q0[SLOTS_IN_FLIGHT][3];
    auto class_sums = [&](int cl) {   // q0: the class's first slots, loaded
        Sum t{};
        add(cl, q0, t);
        for (int K0 = cl + KB_BATCH; K0 < nsum; K0 += KB_BATCH) {
            load_sums(K0, q0);
            add(K0, q0, t);
        }
#pragma unroll
        for (int x = 0; x < 3; x++) sf[cl][x][l] = t.f[x] - t.c[x];
    };
#pragma unroll 1
    for (int cl = w; cl < KB_C; cl += KB_W) {
        unsigned long long mk[SLOTS_IN_FLIGHT];
        Near t{};
        unsigned long long near = 0;
        if constexpr (NEARF) near = near_slots(cl, near0);
        if (cl < nb) {   // a system of few blocks has no slots in the higher classes
            load_masks(cl, near, mk);
            load_sums(cl, q0);
            count(cl, cl, mk, t);
        }
        int batch = 1;
        for (int K0 = cl + KB_BATCH; K0 < nb; K0 += KB_BATCH, batch++) {
            if constexpr (NEARF) near = batch % 6 ? near >> SLOTS_IN_FLIGHT : near_slots(K0, near_bytes(K0));
            load_masks(K0, near, mk);
            count(cl, K0, mk, t);
        }
        s_cnt[cl][l] = t.cn;
        s_nm[cl][l] = t.nm;
        if constexpr (!SUMS_LATE) class_sums(cl);
    }
    __syncthreads();

    // number the block's near entries: ball-major, then class, slot and bit
    int cnt[KB_C], tot = 0;
#pragma unroll
    for (int q = 0; q < KB_C; q++) {
        cnt[q] = s_cnt[q][l];
        tot += cnt[q];
    }
    const int incl = wave_iscan(tot);
    const int total = __builtin_amdgcn_readlane(incl, TB - 1);
    const int b0 = incl - tot, b1 = incl;   // ball l's entries are [b0, b1)

    double n[QW] = {}, npe = 0;
    int ncon = 0, npair = 0;
    for (int r0 = 0;; r0 += KB_T) {
        const int r1 = r0 + KB_T;
        // write this round's entries of (class cl, ball l) for the classes of wavefront w
#pragma unroll 1
        for (int cl = w; cl < KB_C; cl += KB_W) {
            int k = b0, cn = 0;         // (class, ball) entries are [k, k + cn)
#pragma unroll
            for (int q = 0; q < KB_C; q++) {
                if (q < cl) k += cnt[q];
                if (q == cl) cn = cnt[q];
            }
            if (!(cn && k < r1 && k + cn > r0)) continue;
            const int nm = s_nm[cl][l];
            auto put = [&](int K, unsigned long long m) {
                const int e = l | (K << 12);
                auto half = [&](unsigned h, int at) {
                    for (; h; h &= h - 1, k++)
                        if (k >= r0 && k < r1) ent[k - r0] = e | ((at + __builtin_ctz(h)) << 6);
                };
                half((unsigned)m, 0);
                half((unsigned)(m >> 32), 32);
            };
            if (nm <= KB_MC) {
                for (int q = 0; q < nm && k < r1; q++) put(s_mks[cl][q][l], s_mk[cl][q][l]);
            } else {
                for (int K = cl; K < nb && k < r1; K += KB_C)
                    if (!NEARF || a.near[(size_t)blockIdx.x * a.near_stride + K]) put(K, a.nbm[(size_t)K * np + ic]);
            }
        }
        __syncthreads();
        const int t = threadIdx.x;
        if (r0 + t < total) {
            const int e = ent[t];
            const int el = e & (TB - 1), bit = (e >> 6) & (TB - 1), K = e >> 12;
            const NearPair z = near_load(c, a.perm, blockIdx.x * TB + el, off + K * TB + bit);
            double pe;
            res_fl[t] = (unsigned char)near_eval<WRITE>(z, P, &res[0][t], KB_T, pe);
            if (WRITE) res_pe[t] = pe;
        }
        __syncthreads();
        // ball l's entries in this round, in order
        const int k0 = (b0 > r0 ? b0 : r0) - r0, k1 = (b1 < r1 ? b1 : r1) - r0;
#pragma unroll
        for (int u = 0; u < QW; u++) {
            const int q = w + u * NWV;
            if (q < 6) {
                for (int k = k0; k < k1; k++) n[u] = n[u] + res[q][k];
            } else if (q == 6) {
                for (int k = k0; k < k1; k++) {
                    const int fl = res_fl[k];
                    ncon += fl & 1;
                    npair += fl >> 1;
                    if (WRITE) npe = npe + res_pe[k];
                }
            }
        }
        if (r1 >= total) break;
        __syncthreads();   // the next round writes ent and res
    }

    if constexpr (SUMS_LATE) class_sums(w);
    __syncthreads();

    const double dt = P.dt;
#pragma unroll
    for (int u = 0; u < QW; u++) {
        const int q = w + u * NWV;
        if (q >= 6) {
            if (q == 6) {
                // the block's pair energy and pair counts (each pair counted by its ball A)
                const double bpe = WRITE ? wave_sum(far_pe) + wave_sum(npe) : 0.0;
                const int bcc = wave_isum(ncon), bcn = wave_isum(npair);
                if (l == 0) {
                    a.blk_ctr[2 * blockIdx.x] = ctr0 + (unsigned long long)bcc;
                    a.blk_ctr[2 * blockIdx.x + 1] = ctr1 + (unsigned long long)bcn;
                    if (WRITE) {
                        a.e_blk[blockIdx.x * FAST_E_STRIDE] = bpe;
                        a.e_blk[blockIdx.x * FAST_E_STRIDE + 8] = (double)bcc;
                    }
                }
            }
            continue;
        }
        // component q of force (q < 3) or torque, its acceleration, velocity and half step
        const bool lin = q < 3;
        const int x = lin ? q : q - 3;
        double F = n[u];
        if (lin) {
            double s = sf[0][x][l], cmp = 0;
            for (int k = 1; k < KB_C; k++) {
                if (COMP) {
                    const double y = sf[k][x][l] - cmp, t = s + y;
                    cmp = (t - s) - y;
                    s = t;
                } else {
                    s = s + sf[k][x][l];
                }
            }
            F = (s - cmp) + F;
        }
        const int fv = (lin ? VX : WX) + x, fa = (lin ? AX : BX) + x, fh = (lin ? HX : GX) + x;
        const double acc = F / inr[u];
        const double v = a.kick ? h0[u] + .5 * acc * dt : c.at(fv, ic);
        if (valid && !(isfinite(v) && isfinite(x0[u]))) atomicOr(&a.flags[1], 1);
        if (WRITE) {
            fin[q][l] = v;
            if (lin) fin[6 + x][l] = x0[u];
        }
        double xn = x0[u];              // position the next pair pass will read
        double hn = h0[u];
        if (a.drift_next) {
            hn = v + .5 * acc * dt;
            xn = x0[u] + hn * dt;
        }
        if (valid) {
            a.nxt[fv * np + i] = v;
            a.nxt[fa * np + i] = acc;
            a.nxt[fh * np + i] = hn;
            if (lin) {
                a.nxt[(QX + x) * np + i] = a.drift_next ? x0[u] : c.at(QX + x, i);
                a.nxt[(PX + x) * np + i] = xn;
            }
        }
        if (a.drift_next) {
            double* bd = reinterpret_cast<double*>(a.bnd + 2 * blockIdx.x);   // lo, hi
            float* xo = reinterpret_cast<float*>(a.xl + i);
            if (lin) {
                double lo, hi;
                wave_minmax(xn, valid, lo, hi);
                if (l == 0) {
                    bd[x] = lo;
                    bd[4 + x] = hi;
                }
                xo[x] = local_coord(xn, valid, lo, hi, a.L0inv, x == 0 ? l : 0);
            } else if (x == 0) {
                double lo, hi;
                wave_minmax(Rb, valid, lo, hi);
                if (l == 0) {
                    bd[3] = fmax(hi, 0.0);
                    bd[7] = 0;
                }
                xo[3] = valid ? (float)(Rb * a.L0inv) : 0.f;
            }
        }
    }
    if (WRITE) {
        // energy, momenta and the non-finite count; a 64-ball block lies inside one system, so
        // its sums are per system
        __syncthreads();
        const double mi = c.c(MASS, ic), Ii = c.c(MOI, ic);
        const D3 v = d3(fin[0][l], fin[1][l], fin[2][l]), wv = d3(fin[3][l], fin[4][l], fin[5][l]);
        const D3 p0 = d3(fin[6][l], fin[7][l], fin[8][l]);
        for (int k = w; k < 8; k += KB_W) {
            double e;
            if (k == 0) {
                e = .5 * mi * dot(v, v) + .5 * Ii * dot(wv, wv);
            } else if (k < 4) {
                const D3 mv = v * mi;
                e = k == 1 ? mv.x : k == 2 ? mv.y : mv.z;
            } else if (k < 7) {
                const D3 L = cross(p0, v) * mi + wv * Ii;
                e = k == 4 ? L.x : k == 5 ? L.y : L.z;
            } else {
                e = isfinite(v.x) && isfinite(v.y) && isfinite(v.z) && isfinite(wv.x) && isfinite(wv.y) &&
                    isfinite(wv.z) && isfinite(p0.x) && isfinite(p0.y) && isfinite(p0.z) ? 0.0 : 1.0;
            }
            const double sum = wave_sum(valid ? e : 0.0);
            if (l == 0) a.e_blk[blockIdx.x * FAST_E_STRIDE + (k < 7 ? k + 1 : 9)] = sum;
        }
    }
}

// Bounding boxes of the 64-ball blocks (one wavefront per block), for positions that
// did not come from k_ball's drift; DRIFT: after drifting the valid balls (each system with
// its own dt), the start of a call.
template <bool DRIFT>
__global__ __launch_bounds__(TB) void k_bounds(State s, const int4* blk_info, const Phys* sysP, double4* bnd, float4* xl,
                                               double L0inv)
{
    const int l = threadIdx.x;
    const int b = blockIdx.x * TB + l;
    const int4 bi = blk_info[blockIdx.x];
    const bool valid = b - bi.x < bi.y;
    const int bc = valid ? b : bi.x;
    double x = s.f[PX][bc], y = s.f[PY][bc], z = s.f[PZ][bc];
    const double R = s.f[RAD][bc];
    if (DRIFT && valid) {
        const double dt = sysP[bi.w].dt;
        s.f[QX][b] = x;
        s.f[QY][b] = y;
        s.f[QZ][b] = z;
        const double hx = s.f[VX][b] + .5 * s.f[AX][b] * dt;
        const double hy = s.f[VY][b] + .5 * s.f[AY][b] * dt;
        const double hz = s.f[VZ][b] + .5 * s.f[AZ][b] * dt;
        s.f[HX][b] = hx;
        s.f[HY][b] = hy;
        s.f[HZ][b] = hz;
        s.f[GX][b] = s.f[WX][b] + .5 * s.f[BX][b] * dt;
        s.f[GY][b] = s.f[WY][b] + .5 * s.f[BY][b] * dt;
        s.f[GZ][b] = s.f[WZ][b] + .5 * s.f[BZ][b] * dt;
        x = x + hx * dt;
        y = y + hy * dt;
        z = z + hz * dt;
        s.f[PX][b] = x;
        s.f[PY][b] = y;
        s.f[PZ][b] = z;
    }
    double4 lo, hi;
    wave_aabb(x, y, z, R, valid, lo, hi);
    if (l == 0) {
        bnd[2 * blockIdx.x] = lo;
        bnd[2 * blockIdx.x + 1] = hi;
    }
    xl[b] = make_float4(local_coord(x, valid, lo.x, hi.x, L0inv, l), local_coord(y, valid, lo.y, hi.y, L0inv, 0),
                        local_coord(z, valid, lo.z, hi.z, L0inv, 0), valid ? (float)(R * L0inv) : 0.f);
}

}  // namespace fastk
}  // namespace sl
