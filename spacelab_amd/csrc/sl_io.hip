// State read-back: the requested vectors (x, y, z per ball, the caller's layout) are packed by
// a kernel straight into pinned host memory, in pieces of half the staging buffer, and copied
// to the caller's arrays while the next piece is packed.
#include "sl_internal.hpp"

#include <algorithm>
#include <cstring>

namespace sl {

namespace {

struct PackArgs {
    State s;
    int field[MAX_READ];            // first of each vector's three fields
    const int* slot_of;             // caller's slot -> slot of s, NULL: the same
    const int *blk_sys, *sys_off, *sys_n, *sys_first;   // systems (NULL: one, from slot 0)
    int n;                          // balls of the one system
    int slot0, slots;               // this piece: the caller's slots slot0 .. slot0 + slots - 1,
    int ball0, balls;               // which hold the balls ball0 .. ball0 + balls - 1
    double* dst;                    // [vector][ball][xyz]
};

// One thread per component, vectors in grid y: stores run along the caller's array.  Bound
// by the host link and the copy out of the staging buffer: 5 vectors of 129,456 balls (15.5 MB)
// reach the caller's arrays in 0.51 ms (30 GB/s; 4.7 ms when the fields came over whole and
// the host transposed them), 7 vectors of 1,000 balls in 41 us.
__global__ __launch_bounds__(256) void k_pack(PackArgs a)
{
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= 3 * a.slots) return;
    const int c = a.slot0 + e / 3, x = e % 3;
    int ball;
    if (a.blk_sys) {
        const int sy = a.blk_sys[c / FAST_TILE], k = c - a.sys_off[sy];
        if (k >= a.sys_n[sy]) return;
        ball = a.sys_first[sy] + k;
    } else {
        if (c >= a.n) return;
        ball = c;
    }
    const int v = blockIdx.y;
    a.dst[((size_t)v * a.balls + (ball - a.ball0)) * 3 + x] = a.s.f[a.field[v] + x][a.slot_of ? a.slot_of[c] : c];
}

}  // namespace

int stage_alloc(HostStage& hs, size_t bytes)
{
    hs.bytes = bytes / 128 * 128;
    if (hipHostMalloc(&hs.h, hs.bytes, 0) != hipSuccess) return SL_E_HIP;
    if (hipHostGetDevicePointer(reinterpret_cast<void**>(&hs.d), hs.h, 0) != hipSuccess) return SL_E_HIP;
    for (auto& e : hs.ev)
        if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return SL_E_HIP;
    return SL_OK;
}

void stage_free(HostStage& hs)
{
    for (auto& e : hs.ev)
        if (e) (void)hipEventDestroy(e);
    if (hs.h) (void)hipHostFree(hs.h);
    hs = HostStage{};
}

int read_state(HostStage& hs, const State& s, const int* slot_of, const FastLayout& lay, const FastBuffers* fb,
               const int* field, const ReadPart* parts, int nv, hipStream_t st)
{
    PackArgs a{};
    a.s = s;
    a.slot_of = slot_of;
    a.n = lay.n[0];
    if (lay.n_sys > 1) {
        a.blk_sys = fb->blk_sys;
        a.sys_off = fb->sys_off;
        a.sys_n = fb->sys_n;
        a.sys_first = fb->sys_first;
    }
    for (int v = 0; v < nv; v++) a.field[v] = field[v];
    if (nv < 1) return SL_OK;
    // pieces of whole 64-slot blocks, two in flight
    const size_t half = hs.bytes / 2;
    const int per = std::max(1, (int)(half / (nv * 24 * FAST_TILE))) * FAST_TILE;
    if ((size_t)per * nv * 24 > half) return SL_E_STATE;   // the buffer holds at least a block of all vectors twice
    struct Piece {
        int ball0, balls;
    } piece[2];
    int sys = 0, next = 0;          // system of the next slot, next slot
    auto balls_before = [&](int slot) {   // balls in the caller's slots below `slot` (ascending calls)
        while (sys + 1 < lay.n_sys && lay.off[sys + 1] <= slot) sys++;
        return lay.first[sys] + std::min(std::max(slot - lay.off[sys], 0), lay.n[sys]);
    };
    int ball = 0;
    auto pack = [&](int k) -> int {
        a.slot0 = next;
        a.slots = std::min(per, lay.n_used - next);
        a.ball0 = ball;
        next += a.slots;
        ball = next >= lay.n_used ? lay.first[lay.n_sys - 1] + lay.n[lay.n_sys - 1] : balls_before(next);
        a.balls = ball - a.ball0;
        a.dst = reinterpret_cast<double*>(hs.d + (k & 1) * half);
        piece[k & 1] = {a.ball0, a.balls};
        k_pack<<<dim3((3 * a.slots + 255) / 256, nv), 256, 0, st>>>(a);
        return hipGetLastError() == hipSuccess && hipEventRecord(hs.ev[k & 1], st) == hipSuccess ? SL_OK : SL_E_HIP;
    };
    const int pieces = (lay.n_used + per - 1) / per;
    long long done = 0;             // balls of *parts that are out
    if (pack(0)) return SL_E_HIP;
    for (int k = 0; k < pieces; k++) {
        if (k + 1 < pieces && pack(k + 1)) return SL_E_HIP;
        if (hipEventSynchronize(hs.ev[k & 1]) != hipSuccess) return SL_E_HIP;
        const Piece p = piece[k & 1];
        const double* src = reinterpret_cast<const double*>(hs.h + (k & 1) * half);
        for (long long b = 0; b < p.balls;) {
            if (done == parts->balls) {
                parts++;
                done = 0;
            }
            const long long n = std::min<long long>(p.balls - b, parts->balls - done);
            for (int v = 0; v < nv; v++)
                std::memcpy(parts->out[v] + 3 * done, src + 3 * ((size_t)v * p.balls + b), sizeof(double) * 3 * n);
            b += n;
            done += n;
        }
    }
    return SL_OK;
}

}  // namespace sl
