// Surrogate model for collision outcomes: a 4-layer perceptron
//   x (n_in) -> 256 -> 256 -> 256 -> y (n_out), ReLU between layers,
// whose matrix products run on the matrix cores (gfx950's v_mfma_f32_16x16x32_bf16:
// bfloat16 operands, binary32 accumulation, 32 of K per instruction).  Training (forward, loss, backward, Adam) and
// inference are all device kernels; every reduction has a fixed order, so a run is
// reproducible bit for bit.
//
// Two forms, chosen by the layer widths (CHAIN_MAX), with the same results bit for bit:
//   chain   k_chain takes 16 samples through all layers, the loss and the backward
//           products in one launch (every step but the weight gradients is local to a
//           sample), k_wgrad forms the weight and bias gradients of all layers and applies
//           Adam.  Two launches a training step, one an inference; the batch is read from
//           and the results written to pinned host memory by the kernels themselves.
//           Several nets laid out alike share these launches (one grid row per net), and an
//           ensemble's prediction normalises its rows and averages its nets on the device.
//   layers  one launch per product (k_gemm), for wide networks, where a 16-sample
//           workgroup would read each layer's whole weight matrix alone.
//
// Output layout: y[0..2] are the class logits (stick, bounce, fragment), y[3..] are
// regression targets.  Loss per sample: softmax cross-entropy of the logits plus the
// mean squared error of the regression outputs; the batch loss is their mean.
#include "sl_mlp_host.hpp"
#include "spacelab/sl_api.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <new>
#include <string>
#include <type_traits>

namespace {

using bf16 = unsigned short;
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));

constexpr int NL = 4;          // layers
constexpr int GM = 32;         // GEMM block tile rows
constexpr int GN = 32;         // GEMM block tile columns
constexpr int GK = 64;         // GEMM K step staged in LDS
constexpr int NCLS = 3;

// Round to nearest even (the hardware's conversion).
__device__ __forceinline__ bf16 to_bf16(float f) { return __builtin_bit_cast(bf16, (__bf16)f); }

// C[M][N] = op(A)[M][K] * op(B)[K][N] (+ bias[N]) with bfloat16 operands and binary32
// accumulation.  op(A)(m, k) = TA ? A[k * lda + m] : A[m * lda + k]; op(B)(k, n) =
// TB ? B[n * ldb + k] : B[k * ldb + n].  Optional ReLU; the result is stored in binary32
// (C) and/or bfloat16 (Cb).  A 256-thread block computes a 32 x 32 tile: wavefront w
// owns the 16 x 16 quarter (w / 2, w % 2), one v_mfma_f32_16x16x32_bf16 per 32 of K
// (lane l: row or column l % 16, K values 8 (l / 16) .. 8 (l / 16) + 7 of the step, the
// same K values for both operands).  Operand tiles of GK = 64 along K are staged through
// LDS (zero fill outside the matrices); global reads run along each matrix's contiguous
// index, and both tiles are stored K-contiguous so each lane reads its eight K values as
// one 16-byte word.  The small output tile keeps many workgroups in flight for the
// 256-wide layers.
//
// With csum, the blocks of the first row of tiles also form the column sums of the
// binary32 matrix csrc[K][ldcs] over its K rows for their GN columns (the bias gradient
// beside the weight gradient X^T dZ): 8 row phases per column, phase p adding rows p,
// p + 8, ... in order, then the phases added in order.
template <bool TA, bool TB>
__global__ __launch_bounds__(256) void k_gemm(int M, int N, int K, const bf16* A, int lda, const bf16* B, int ldb,
                                              float* C, int ldc, bf16* Cb, int ldcb, const float* bias, int relu,
                                              const float* csrc, int ldcs, float* csum)
{
    __shared__ __attribute__((aligned(16))) bf16 As[GM][GK + 8];   // [m][k]
    __shared__ __attribute__((aligned(16))) bf16 Bt[GN][GK + 8];   // [n][k]
    const int tid = threadIdx.x, w = tid / 64, l = tid % 64;
    const int m0 = blockIdx.y * GM, n0 = blockIdx.x * GN;
    const int wm = (w / 2) * 16, wn = (w % 2) * 16;
    float4_t acc = float4_t{0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < K; k0 += GK) {
        for (int e = tid; e < GM * GK; e += 256) {
            int r, c;   // r: m within the tile, c: k within the step
            if (TA) {
                c = e / GM;
                r = e % GM;
            } else {
                r = e / GK;
                c = e % GK;
            }
            const int gm = m0 + r, gk = k0 + c;
            bf16 v = 0;
            if (gm < M && gk < K) v = TA ? A[(size_t)gk * lda + gm] : A[(size_t)gm * lda + gk];
            As[r][c] = v;
        }
        for (int e = tid; e < GK * GN; e += 256) {
            int r, c;   // r: k within the step, c: n within the tile
            if (TB) {
                c = e / GK;
                r = e % GK;
            } else {
                r = e / GN;
                c = e % GN;
            }
            const int gk = k0 + r, gn = n0 + c;
            bf16 v = 0;
            if (gk < K && gn < N) v = TB ? B[(size_t)gn * ldb + gk] : B[(size_t)gk * ldb + gn];
            Bt[c][r] = v;
        }
        __syncthreads();
        const int row = wm + (l % 16), col = wn + (l % 16);
#pragma unroll
        for (int kk = 0; kk < GK; kk += 32) {
            const int kq = kk + 8 * (l / 16);
            const bf16x8_t a = *reinterpret_cast<const bf16x8_t*>(&As[row][kq]);
            const bf16x8_t b = *reinterpret_cast<const bf16x8_t*>(&Bt[col][kq]);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
        }
        __syncthreads();
    }
    if (csum && blockIdx.y == 0) {
        __shared__ float part[8][GN];
        const int cl = tid % GN, ph = tid / GN;   // 8 phases of GN columns
        const int c = n0 + cl;
        float sum = 0.f;
        if (c < N) {
            // the loads run ahead of the (ordered) additions
#pragma unroll 8
            for (int r = ph; r < K; r += 8) sum += csrc[(size_t)r * ldcs + c];
        }
        part[ph][cl] = sum;
        __syncthreads();
        if (ph == 0 && c < N) {
            float v = part[0][cl];
            for (int q = 1; q < 8; q++) v += part[q][cl];
            csum[c] = v;
        }
    }
    for (int r = 0; r < 4; r++) {
        const int row = m0 + wm + 4 * (l / 16) + r;
        const int col = n0 + wn + (l % 16);
        if (row >= M || col >= N) continue;
        float v = acc[r];
        if (bias) v += bias[col];
        if (relu && v < 0.f) v = 0.f;
        if (C) C[(size_t)row * ldc + col] = v;
        if (Cb) Cb[(size_t)row * ldcb + col] = to_bf16(v);
    }
}

// Rows of x (n_in wide) into a zero-padded bfloat16 matrix ld wide.
__global__ void k_pack_input(int B, int n_in, int ld, const float* x, bf16* xb)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= B * ld) return;
    const int r = i / ld, c = i % ld;
    xb[i] = c < n_in ? to_bf16(x[(size_t)r * n_in + c]) : (bf16)0;
}

// Loss of one sample and its gradient with respect to the outputs (in place over the
// outputs z[0 .. ldy)): CE(softmax(z[0..2]), c) + mean_k (z[3+k] - reg[k])^2, gradient
// scaled by invB.
__device__ __forceinline__ float sample_loss(float* z, int n_out, int ldy, int c, const float* reg, float invB)
{
    float mx = z[0];
    for (int k = 1; k < NCLS; k++) mx = fmaxf(mx, z[k]);
    float se = 0.f, p[NCLS];
    for (int k = 0; k < NCLS; k++) {
        p[k] = expf(z[k] - mx);
        se += p[k];
    }
    float loss = logf(se) + mx - z[c];
    const int nr = n_out - NCLS;
    for (int k = 0; k < NCLS; k++) z[k] = (p[k] / se - (k == c ? 1.f : 0.f)) * invB;
    for (int k = 0; k < nr; k++) {
        const float d = z[NCLS + k] - reg[k];
        loss += d * d / (float)nr;
        z[NCLS + k] = 2.f * d / (float)nr * invB;
    }
    for (int k = n_out; k < ldy; k++) z[k] = 0.f;
    return loss;
}

// One thread per sample; the gradient goes to dy (binary32) and dyb (bfloat16).
__global__ void k_loss(int B, int n_out, int ldy, const float* y, const int* cls, const float* reg, float* dy,
                       bf16* dyb, float* loss_s)
{
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= B) return;
    float* g = dy + (size_t)b * ldy;
    for (int k = 0; k < ldy; k++) g[k] = y[(size_t)b * ldy + k];
    loss_s[b] = sample_loss(g, n_out, ldy, cls[b], reg + (size_t)b * (n_out - NCLS), 1.0f / (float)B);
    for (int k = 0; k < ldy; k++) dyb[(size_t)b * ldy + k] = to_bf16(g[k]);
}

// dZ = dH * (Z > 0): ReLU backward, in binary32 and bfloat16.
__global__ void k_relu_back(int n, const float* z, float* dz, bf16* dzb)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float g = z[i] > 0.f ? dz[i] : 0.f;
    dz[i] = g;
    dzb[i] = to_bf16(g);
}

// Adam (Kingma & Ba 2015) on binary32 master weights: the step's constants, and the update
// of one value.
struct Adam {
    float lr, b1, b2, eps, c1, c2;
};

__device__ __forceinline__ float adam_value(const Adam& a, float w, float g, float& m, float& v)
{
    const float mi = a.b1 * m + (1.f - a.b1) * g;
    const float vi = a.b2 * v + (1.f - a.b2) * g * g;
    m = mi;
    v = vi;
    return w - a.lr * (mi / a.c1) / (sqrtf(vi / a.c2) + a.eps);
}

__global__ void k_adam(int n, float* w, bf16* wb, const float* g, float* m, float* v, Adam a)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float wi = adam_value(a, w[i], g[i], m[i], v[i]);
    w[i] = wi;
    if (wb) wb[i] = to_bf16(wi);
}

// Softmax probabilities and predictive entropy (nats) of one sample's class logits.
__device__ __forceinline__ float sample_predict(const float* z, float* prob)
{
    float mx = z[0];
    for (int k = 1; k < NCLS; k++) mx = fmaxf(mx, z[k]);
    float p[NCLS], se = 0.f;
    for (int k = 0; k < NCLS; k++) {
        p[k] = expf(z[k] - mx);
        se += p[k];
    }
    float h = 0.f;
    for (int k = 0; k < NCLS; k++) {
        p[k] /= se;
        prob[k] = p[k];
        if (p[k] > 0.f) h -= p[k] * logf(p[k]);
    }
    return h;
}

__global__ void k_predict(int B, int ldy, const float* y, float* prob, float* ent)
{
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= B) return;
    ent[b] = sample_predict(y + (size_t)b * ldy, prob + (size_t)b * NCLS);
}

// ---- the chain form -------------------------------------------------------------------

constexpr int CHAIN_ROWS = 16;           // samples per workgroup: one MFMA tile of rows
// Widest (padded) layer the chain form takes: two column tiles per wavefront, the ReLU masks
// in one register, the activations in LDS.  Measured there (21-W-W-W-9, us per call, chain /
// layers): W 512 batch 16 training 74 / 253, batch 256 78 / 340, batch 4096 169 / 1622,
// inference 35 / 152, 36 / 180, 52 / 262; W 128 batch 256 38 / 226 and 27 / 135.
constexpr int CHAIN_MAX = 512;
constexpr int CHAIN_WAVES = 16;          // most wavefronts per workgroup
constexpr int CHAIN_LD = CHAIN_MAX + 8;  // row stride of the activations in LDS: 16-byte reads of 16 rows, no conflicts
constexpr int KF = 8;                    // weight fragments (32 of K each) a lane holds at once

// Members of an ensemble that one launch carries through the same pass (grid y): nets of the
// same widths and largest batch are laid out alike, so a member's pointer is the first
// member's, moved by the distance between their allocations.  One net has too few workgroups
// (16 at batch 256) and too short a pass for a launch: a training step of four nets takes the
// device 33 us together and 27 us for one alone; driven one by one each cost 56 us with its
// launches and its wait.  (21-256-256-256-9, batch 256, 4096 rows, one epoch of four nets:
// 3.6 -> 1.5 ms, 1.2 with the next batch gathered meanwhile; 10,000 rows through the four 1.03
// -> 0.76 ms.)
constexpr int MEMBERS = 16;
struct Moved {
    long long pool, stage, x;   // bytes: device pool, pinned buffer, input rows
};
template <class T>
__device__ __forceinline__ T* moved(T* p, long long by)
{
    using C = std::conditional_t<std::is_const_v<T>, const char, char>;
    return reinterpret_cast<T*>(reinterpret_cast<C*>(p) + by);
}

struct ChainArgs {
    Moved at[MEMBERS];
    int B, n_in, n_out;
    int ld[NL + 1];                 // padded widths: input, hidden layers, output
    const float* x;                 // [B][n_in]
    const int* cls;
    const float* reg;               // [B][n_out - 3]
    const bf16* Wf[NL];             // forward weights (K inputs, N outputs) as fragments
    const bf16* Wr[NL];             // backward ones (K outputs, N inputs)
    const float* b[NL];
    // training: inputs and output gradients of every layer for k_wgrad, feature-major
    // ([feature][ldb], K = sample contiguous); the gradients in binary32 too ([B][ld])
    bf16* Ht[NL];
    bf16* dZt[NL];
    float* dZ[NL];
    int ldb;
    float* loss;                    // [B]
    float *y, *prob, *ent;          // inference: [B][n_out], [B][3], [B]
};

// Weights for the chain are kept in the order the MFMA fragments want them: for a product
// with K inputs and N outputs, 1 KB per (16 outputs, 32 inputs), lane l's eight values (output
// l % 16, inputs 8 (l / 16) .. + 7 of the 32, zero past K) at 16 l bytes, the tiles of
// 16 outputs one after another.  A wavefront's load is then 1 KB in a row; with the rows
// of a plain [out][in] matrix it was 16 pieces of 64 bytes, and a layer of 256 x 256
// took 4.3 us to reach a CU.  frag_at: element (k, n) of such a matrix of ks steps.
__device__ __forceinline__ size_t frag_at(int k, int n, int ks)
{
    return ((size_t)(n / 16 * ks + k / 32) * 64 + k % 32 / 8 * 16 + n % 16) * 8 + k % 8;
}

__host__ __device__ inline int k_steps(int K) { return (K + 31) / 32; }

// The fragments of output tile `tile`, steps s0 .. s0 + F - 1 (the last step again past the
// end: every path sends the same number of loads, which lets the compiler wait for one
// product's loads while the next one's stay in flight).
template <int F>
__device__ __forceinline__ void load_frags(bf16x8_t (&wf)[KF], const bf16* mat, int tile, int ks, int s0)
{
    const bf16x8_t* p = reinterpret_cast<const bf16x8_t*>(mat) + (size_t)tile * ks * 64 + threadIdx.x % 64;
#pragma unroll
    for (int s = 0; s < F; s++) wf[s] = p[min(s0 + s, ks - 1) * 64];
}

// One wavefront's 16 x 16 tile of (16 samples in LDS) x (weights): wf holds the first F
// steps' fragments, loaded ahead by the caller.  The K values of a lane are those of
// k_gemm and the steps ascend, so the sums have k_gemm's bits.
template <int F>
__device__ __forceinline__ float4_t chain_tile(const bf16 (*A)[CHAIN_LD], bf16x8_t (&wf)[KF], const bf16* mat,
                                               int tile, int ks)
{
    const int l = threadIdx.x % 64;
    const bf16* row = &A[l % 16][8 * (l / 16)];
    float4_t acc = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < F; s++) {
        if (s >= ks) break;
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8_t*>(row + 32 * s), wf[s], acc, 0, 0, 0);
    }
    for (int s0 = F; s0 < ks; s0 += F) {
        load_frags<F>(wf, mat, tile, ks, s0);
#pragma unroll
        for (int s = 0; s < F; s++) {
            if (s0 + s >= ks) break;
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8_t*>(row + 32 * (s0 + s)), wf[s],
                                                          acc, 0, 0, 0);
        }
    }
    return acc;
}

// Workgroup barrier for data passed through LDS only: unlike __syncthreads it leaves
// global loads (the next layers' weights) in flight.
__device__ __forceinline__ void lds_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Four consecutive samples of one feature as bfloat16, at sample offset q of its row.
__device__ __forceinline__ void store4(bf16* row, int q, const float (&v)[4])
{
    typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
    *reinterpret_cast<bf16x4_t*>(row + q) = bf16x4_t{(__bf16)v[0], (__bf16)v[1], (__bf16)v[2], (__bf16)v[3]};
}

// Forward pass of 16 samples through every layer (and, TRAIN, loss and backward products
// down to the first hidden layer's gradient), one workgroup.  Wavefront w makes the
// column tiles w, w + nw of each layer; the activations pass from layer to layer
// through LDS, one barrier each.  A lane that makes (sample, feature) forward makes it
// backward too, so the ReLU masks stay in registers.
// Bound by latency, not by throughput: 16 workgroups at batch 256, each a chain of four
// (training: seven) products whose weights come from L2 and beyond.  So the weights of the
// next two products are always on the way: two fragment buffers, each refilled as soon
// as its product is done; biases, labels and targets are fetched at the start, because a
// load waits for all those sent before it.  Measured at 21-256-256-256-9, batch 256: 20.9
// us training (5 us of it the batch's way from host memory, 2 us a product), 15.4 us
// inference; the products one by one took 17 us each forward, 13 and 18 us backward.
// F0, FL: fragments held of the first product's and the first backward product's K (1 when
// the network has at most 32 inputs or outputs, else KF).
template <bool TRAIN, int F0, int FL>
__global__ __launch_bounds__(CHAIN_WAVES * 64) void k_chain(ChainArgs a)
{
    __shared__ __attribute__((aligned(16))) bf16 act[2][CHAIN_ROWS][CHAIN_LD];
    __shared__ float yf[CHAIN_ROWS][CHAIN_MAX + 1];
    __shared__ float rg[TRAIN ? CHAIN_ROWS : 1][TRAIN ? CHAIN_MAX : 1];   // regression targets
    __shared__ float bs[NL][CHAIN_MAX];                                   // biases
    const Moved at = a.at[blockIdx.y];
    const int t = threadIdx.x, nt = blockDim.x, nw = nt / 64;
    const int w = __builtin_amdgcn_readfirstlane(t / 64), l = t % 64;
    const int m0 = blockIdx.x * CHAIN_ROWS;
    const int r0 = 4 * (l / 16), cl = l % 16;     // this lane's rows r0 .. r0 + 3 and column within a tile
    bf16x8_t wf[2][KF];
    // Product p of the chain: 0 .. NL - 1 forward, then backward through layers NL - 1 .. 1.
    // ask(p) sends for its first tile's fragments (a wavefront without a tile: the last one's).
    auto ask = [&](auto pc) {
        constexpr int p = decltype(pc)::value;
        constexpr int k = p < NL ? p : 2 * NL - 1 - p;
        const bf16* mat = p < NL ? moved(a.Wf[k], at.pool) : moved(a.Wr[k], at.pool);
        const int K = p < NL ? a.ld[k] : a.ld[k + 1], N = p < NL ? a.ld[k + 1] : a.ld[k];
        constexpr int F = p == 0 ? F0 : p == NL ? FL : KF;
        load_frags<F>(wf[p & 1], mat, min(w, N / 16 - 1), k_steps(K), 0);
    };
    ask(std::integral_constant<int, 0>{});
    ask(std::integral_constant<int, 1>{});
    // the input rows, padded with zeros to a multiple of 32, the labels and the targets
    int cls = 0;
    if (TRAIN && t < CHAIN_ROWS && m0 + t < a.B) cls = moved(a.cls, at.stage)[m0 + t];
#pragma unroll 1
    for (int r = w; r < CHAIN_ROWS; r += nw) {
        const size_t b = m0 + r;
        const bool in = m0 + r < a.B;
#pragma unroll 1
        for (int c = l; c < 32 * k_steps(a.ld[0]); c += 64)
            act[0][r][c] = to_bf16(in && c < a.n_in ? moved(a.x, at.x)[b * a.n_in + c] : 0.f);
        if (TRAIN && in)
#pragma unroll 1
            for (int c = l; c < a.n_out - NCLS; c += 64) rg[r][c] = moved(a.reg, at.stage)[b * (a.n_out - NCLS) + c];
    }
    for (int k = 0; k < NL; k++)
#pragma unroll 1
        for (int c = t; c < a.ld[k + 1]; c += nt) bs[k][c] = moved(a.b[k], at.pool)[c];
    lds_barrier();
    if (TRAIN)
#pragma unroll 1
        for (int e = t; e < 4 * a.ld[0]; e += nt) {
            const int c = e / 4, q = 4 * (e % 4);
            const unsigned lo = (unsigned)act[0][q][c] | (unsigned)act[0][q + 1][c] << 16;
            const unsigned hi = (unsigned)act[0][q + 2][c] | (unsigned)act[0][q + 3][c] << 16;
            *reinterpret_cast<uint2*>(moved(a.Ht[0], at.pool) + (size_t)c * a.ldb + m0 + q) = make_uint2(lo, hi);
        }
    unsigned mask = 0;   // 4 bits per hidden layer and tile of this wavefront: the outputs above 0
    auto fwd = [&](auto kc) {
        constexpr int k = decltype(kc)::value;
        constexpr bool last = k == NL - 1;
        constexpr int F = k == 0 ? F0 : KF;
        const int N = a.ld[k + 1], ks = k_steps(a.ld[k]);
        auto tile = [&](int n0, int ti) {
            const float bias = bs[k][n0 + cl];
            const float4_t acc = chain_tile<F>(act[k & 1], wf[k & 1], moved(a.Wf[k], at.pool), n0 / 16, ks);
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                v[r] = acc[r] + bias;
                if (!last && v[r] < 0.f) v[r] = 0.f;
            }
            if (last) {
#pragma unroll
                for (int r = 0; r < 4; r++) yf[r0 + r][n0 + cl] = v[r];
            } else {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    act[(k + 1) & 1][r0 + r][n0 + cl] = to_bf16(v[r]);
                    if (TRAIN) {
                        if (v[r] > 0.f) mask |= 1u << (8 * k + 4 * ti + r);
                        if (m0 + r0 + r >= a.B) v[r] = 0.f;   // rows past the batch: nothing for k_wgrad
                    }
                }
                if (TRAIN) store4(moved(a.Ht[last ? 0 : k + 1], at.pool) + (size_t)(n0 + cl) * a.ldb, m0 + r0, v);
            }
        };
        if (16 * w < N) tile(16 * w, 0);
        if (16 * (w + nw) < N) {   // at most two tiles: CHAIN_MAX / 16 / CHAIN_WAVES
            load_frags<F>(wf[k & 1], moved(a.Wf[k], at.pool), w + nw, ks, 0);
            tile(16 * (w + nw), 1);
        }
        if (!last && (N & 16) && w == nw - 1)
            for (int r = 0; r < 4; r++) act[(k + 1) & 1][r0 + r][N + cl] = 0;
        if constexpr (k + 2 < (TRAIN ? 2 * NL - 1 : NL)) ask(std::integral_constant<int, k + 2>{});
        lds_barrier();
    };
    fwd(std::integral_constant<int, 0>{});
    fwd(std::integral_constant<int, 1>{});
    fwd(std::integral_constant<int, 2>{});
    fwd(std::integral_constant<int, 3>{});
    const int ldy = a.ld[NL];
    if constexpr (!TRAIN) {
#pragma unroll 1
        for (int r = w; r < CHAIN_ROWS; r += nw)
            if (m0 + r < a.B)
#pragma unroll 1
                for (int c = l; c < a.n_out; c += 64) moved(a.y, at.stage)[(size_t)(m0 + r) * a.n_out + c] = yf[r][c];
        if (t < CHAIN_ROWS && m0 + t < a.B) {
            float p[NCLS];
            moved(a.ent, at.stage)[m0 + t] = sample_predict(yf[t], p);
            for (int k = 0; k < NCLS; k++) moved(a.prob, at.stage)[(size_t)(m0 + t) * NCLS + k] = p[k];
        }
        return;
    }
    // loss and output gradient (the forward products left act[0] free: NL is even)
    if (t < CHAIN_ROWS) {
        const int b = m0 + t;
        if (b < a.B)
            moved(a.loss, at.stage)[b] = sample_loss(yf[t], a.n_out, ldy, cls, rg[t], 1.0f / (float)a.B);
        else
            for (int k = 0; k < ldy; k++) yf[t][k] = 0.f;
    }
    lds_barrier();
#pragma unroll 1
    for (int r = w; r < CHAIN_ROWS; r += nw)
#pragma unroll 1
        for (int c = l; c < 32 * k_steps(ldy); c += 64) {
            const float g = c < ldy ? yf[r][c] : 0.f;
            act[0][r][c] = to_bf16(g);
            if (c < ldy && m0 + r < a.B) moved(a.dZ[NL - 1], at.pool)[(size_t)(m0 + r) * ldy + c] = g;
        }
#pragma unroll 1
    for (int e = t; e < 4 * ldy; e += nt) {
        const int c = e / 4, q = 4 * (e % 4);
        const float v[4] = {yf[q][c], yf[q + 1][c], yf[q + 2][c], yf[q + 3][c]};
        store4(moved(a.dZt[NL - 1], at.pool) + (size_t)c * a.ldb, m0 + q, v);
    }
    lds_barrier();
    auto bwd = [&](auto pc) {
        constexpr int p = decltype(pc)::value;
        constexpr int k = 2 * NL - 1 - p;             // the layer gone back through
        constexpr int F = p == NL ? FL : KF;
        constexpr int cur = p & 1;                    // act[0] holds the output gradient: NL is even
        const int N = a.ld[k], ks = k_steps(a.ld[k + 1]);
        auto tile = [&](int n0, int ti) {
            const float4_t acc = chain_tile<F>(act[cur], wf[p & 1], moved(a.Wr[k], at.pool), n0 / 16, ks);
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const bool in = m0 + r0 + r < a.B;
                v[r] = in && ((mask >> (8 * (k - 1) + 4 * ti + r)) & 1u) ? acc[r] : 0.f;
                if (in) moved(a.dZ[k - 1], at.pool)[(size_t)(m0 + r0 + r) * N + n0 + cl] = v[r];
                act[cur ^ 1][r0 + r][n0 + cl] = to_bf16(v[r]);
            }
            store4(moved(a.dZt[k - 1], at.pool) + (size_t)(n0 + cl) * a.ldb, m0 + r0, v);
        };
        if (16 * w < N) tile(16 * w, 0);
        if (16 * (w + nw) < N) {
            load_frags<F>(wf[p & 1], moved(a.Wr[k], at.pool), w + nw, ks, 0);
            tile(16 * (w + nw), 1);
        }
        if ((N & 16) && w == nw - 1)
            for (int r = 0; r < 4; r++) act[cur ^ 1][r0 + r][N + cl] = 0;
        if constexpr (p + 2 < 2 * NL - 1) ask(std::integral_constant<int, p + 2>{});
        lds_barrier();
    };
    bwd(std::integral_constant<int, NL>{});
    bwd(std::integral_constant<int, NL + 1>{});
    bwd(std::integral_constant<int, NL + 2>{});
}

// Weight and bias gradients of every layer from k_chain's feature-major buffers, then
// Adam (STEP) or the gradients stored.  One wavefront per 16 x 16 tile of a layer's H^T dZ
// (K = the batch, ascending: k_gemm's sums), both operands read as 16-byte fragments straight
// from memory, KF steps in flight; after the weight tiles, one workgroup per 32 columns
// of a layer's bias (8 row phases per column as in k_gemm).
// Bound by latency: 560 tiles of 8 steps at batch 256.  The moments and weights a
// tile updates are loaded beside its first operands.  Measured at 21-256-256-256-9, batch
// 256: 5.6 us; four products of 18 us and eight Adam launches of 2.4 us before.
struct WgradArgs {
    int B, ldb;
    int ld[NL + 1];
    int tile0[NL + 1];              // first weight tile of each layer, total at the end
    int bias0[NL + 1];              // first bias workgroup of each layer
    int wblocks;                    // workgroups of weight tiles
    const bf16* Ht[NL];
    const bf16* dZt[NL];
    const float* dZ[NL];
    float *W[NL], *mW[NL], *vW[NL], *gW[NL];
    bf16 *Wf[NL], *Wr[NL];
    float *b[NL], *mb[NL], *vb[NL], *gb[NL];
    long long pool[MEMBERS];        // as in Moved
    Adam adam[MEMBERS];
};

template <bool STEP>
__global__ __launch_bounds__(256) void k_wgrad(WgradArgs a)
{
    const int tid = threadIdx.x;
    const long long at = a.pool[blockIdx.y];
    const Adam adam = a.adam[blockIdx.y];
    if ((int)blockIdx.x >= a.wblocks) {
        __shared__ float part[8][32];
        const int q = blockIdx.x - a.wblocks;
        int k = 0;
        while (k + 1 < NL && q >= a.bias0[k + 1]) k++;
        const int N = a.ld[k + 1];
        const int cl = tid % 32, ph = tid / 32;
        const int c = (q - a.bias0[k]) * 32 + cl;
        float sum = 0.f;
        if (c < N) {
            const float* src = moved(a.dZ[k], at) + c;
#pragma unroll 8
            for (int r = ph; r < a.B; r += 8) sum += src[(size_t)r * N];
        }
        part[ph][cl] = sum;
        __syncthreads();
        if (ph == 0 && c < N) {
            float g = part[0][cl];
            for (int p = 1; p < 8; p++) g += part[p][cl];
            if (STEP)
                moved(a.b[k], at)[c] = adam_value(adam, moved(a.b[k], at)[c], g, moved(a.mb[k], at)[c], moved(a.vb[k], at)[c]);
            else
                moved(a.gb[k], at)[c] = g;
        }
        return;
    }
    const int w = __builtin_amdgcn_readfirstlane(tid / 64), l = tid % 64;
    const int tile = blockIdx.x * 4 + w;
    if (tile >= a.tile0[NL]) return;
    int k = 0;
    while (k + 1 < NL && tile >= a.tile0[k + 1]) k++;
    const int K = a.ld[k], N = a.ld[k + 1];       // the layer's input and output widths
    const int nt = N / 16;
    const int i0 = (tile - a.tile0[k]) / nt * 16, o0 = (tile - a.tile0[k]) % nt * 16;
    const int out = o0 + l % 16, in0 = i0 + 4 * (l / 16);
    float wv[4], mv[4], vv[4];
    if (STEP) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const size_t e = (size_t)(in0 + r) * N + out;
            wv[r] = moved(a.W[k], at)[e];
            mv[r] = moved(a.mW[k], at)[e];
            vv[r] = moved(a.vW[k], at)[e];
        }
    }
    const bf16* ha = moved(a.Ht[k], at) + (size_t)(i0 + l % 16) * a.ldb + 8 * (l / 16);
    const bf16* zb = moved(a.dZt[k], at) + (size_t)(o0 + l % 16) * a.ldb + 8 * (l / 16);
    // ldb covers the batch in steps of 32; rows past it in k_chain's last 16 are zeros, and
    // the 16 after those are not read
    const int Bp = (a.B + CHAIN_ROWS - 1) / CHAIN_ROWS * CHAIN_ROWS;
    float4_t acc = float4_t{0.f, 0.f, 0.f, 0.f};
    for (int b0 = 0; b0 < Bp; b0 += 32 * KF) {
        bf16x8_t ah[KF], bz[KF];
#pragma unroll
        for (int s = 0; s < KF; s++) {
            const int q = b0 + 32 * s;
            if (q + 8 * (l / 16) < Bp) {
                ah[s] = *reinterpret_cast<const bf16x8_t*>(ha + q);
                bz[s] = *reinterpret_cast<const bf16x8_t*>(zb + q);
            } else {
                ah[s] = bf16x8_t{};
                bz[s] = bf16x8_t{};
            }
        }
#pragma unroll
        for (int s = 0; s < KF; s++)
            if (b0 + 32 * s < Bp) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[s], bz[s], acc, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const size_t e = (size_t)(in0 + r) * N + out;
        if (STEP) {
            wv[r] = adam_value(adam, wv[r], acc[r], mv[r], vv[r]);
            moved(a.W[k], at)[e] = wv[r];
            moved(a.mW[k], at)[e] = mv[r];
            moved(a.vW[k], at)[e] = vv[r];
            moved(a.Wr[k], at)[frag_at(out, in0 + r, k_steps(N))] = to_bf16(wv[r]);
        } else {
            moved(a.gW[k], at)[e] = acc[r];
        }
    }
    if (STEP) store4(moved(a.Wf[k], at) + frag_at(in0, out, k_steps(K)), 0, wv);
}

// Rows of descriptors to the nets' inputs, (x - mean) / std in T, rounded to binary32.
template <class T>
__global__ __launch_bounds__(256) void k_normalise(int n, int n_in, const T* x, const T* mean, const T* std, float* out)
{
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e < n * n_in) out[e] = (float)((x[e] - mean[e % n_in]) / std[e % n_in]);
}

// An ensemble's answer for a row, one thread each: the members' class probabilities and
// regression outputs added in binary64 in their order and divided by their number, the most
// probable class (the first of equals; the first NaN, if any) and the entropy.
// With k_normalise in front and the nets' outputs kept on the device: 10,000 rows through four
// nets 763 -> 246 us (the host's normalising, adding and entropy were three quarters of it);
// binary32 rows 205 us.
struct EnsembleArgs {
    long long at[MEMBERS];   // members' outputs, as in Moved
    int n, B, n_out;
    const float *y, *prob;   // [B][n_out], [B][3]
    int* cls;
    float* reg;              // [B][n_out - 3]
    double *p, *ent;         // [B][3], [B]
};
__global__ __launch_bounds__(64) void k_ensemble(EnsembleArgs a)
{
    const int b = blockIdx.x * 64 + threadIdx.x;
    if (b >= a.B) return;
    const int nr = a.n_out - NCLS;
    double p[NCLS];
    for (int c = 0; c < NCLS; c++) {
        double s = 0;
        for (int j = 0; j < a.n; j++) s = s + (double)moved(a.prob, a.at[j])[(size_t)b * NCLS + c];
        p[c] = s / (double)a.n;
        a.p[(size_t)b * NCLS + c] = p[c];
    }
    for (int k = 0; k < nr; k++) {
        double s = 0;
        for (int j = 0; j < a.n; j++) s = s + (double)moved(a.y, a.at[j])[(size_t)b * a.n_out + NCLS + k];
        a.reg[(size_t)b * nr + k] = (float)(s / (double)a.n);
    }
    int best = 0;
    double h = 0;
    for (int c = 0; c < NCLS; c++) {
        if (!(p[best] != p[best]) && (p[c] > p[best] || p[c] != p[c])) best = c;
        h = h + p[c] * ::log(p[c] > 0 ? p[c] : 1.0);
    }
    a.cls[b] = best;
    a.ent[b] = -h;
}

// bfloat16 copies of one layer's weights: Wb in W's layout (layer form), or Wf and Wr as
// fragments (chain form; the parts past the layer's widths stay as they are).
__global__ void k_weights_bf16(int K, int N, const float* W, bf16* Wb, bf16* Wf, bf16* Wr)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= K * N) return;
    const bf16 v = to_bf16(W[e]);
    if (Wb) {
        Wb[e] = v;
        return;
    }
    Wf[frag_at(e / N, e % N, k_steps(K))] = v;
    Wr[frag_at(e % N, e / N, k_steps(N))] = v;
}

struct Layer {
    int in, out, ldin, ldout;   // logical and padded widths
    float* W = nullptr;         // [in][out] binary32 master (padded rows/cols are zero)
    bf16* Wb = nullptr;         // bfloat16 copy (layer form)
    bf16 *Wf = nullptr, *Wr = nullptr;   // the same as fragments, forward and backward (chain form)
    float* b = nullptr;         // [out]
    float *gW = nullptr, *gb = nullptr;
    float *mW = nullptr, *vW = nullptr, *mb = nullptr, *vb = nullptr;
};

}  // namespace

struct sl_mlp {
    int device = 0;
    int n_in = 0, width = 0, n_out = 0, max_batch = 0;
    bool chain = false;              // the chain form (layer widths up to CHAIN_MAX)
    hipStream_t stream = nullptr;
    Layer L[NL];
    // One device allocation: the parameters (per layer W then b, padded), their gradients,
    // both moments (each in the same layout, n_flat floats), the bfloat16 copies and the
    // activations.
    char* pool = nullptr;
    size_t n_flat = 0;
    float *params = nullptr, *grads = nullptr, *moments = nullptr;
    // One pinned host allocation (sl::pinned_bytes): a batch and its results in the chain form
    // (the kernels read and write it), the losses in the layer form, the padded parameters, or a
    // piece of them, during exchanges.
    char* stage = nullptr;
    size_t stage_bytes = 0;
    char* stage_dev = nullptr;       // its device address
    hipEvent_t half[2] = {};         // an ensemble's batches in flight
    // chain form: activations and output gradients, feature-major, and the gradients in binary32
    bf16 *Ht[NL] = {}, *dZt[NL] = {};
    int ldb = 0;
    // layer form: activations Z (post-activation, binary32) and H (bfloat16) per layer
    bf16* xb = nullptr;              // packed input [max_batch][ld0]
    float* Z[NL] = {};
    bf16* Hb[NL] = {};
    float* dZ[NL] = {};              // (both forms)
    bf16* dZb[NL] = {};
    float *xin = nullptr, *reg = nullptr, *loss_s = nullptr, *prob = nullptr, *ent = nullptr;   // (xin, prob, ent: both forms)
    float* yout = nullptr;           // chain form, ensembles: outputs
    int* cls = nullptr;
    long long t = 0;                 // Adam step
    std::string err;
};

namespace {

int pad16(int n) { return (n + 15) / 16 * 16; }

int mlp_err(sl_mlp* m, int code, const char* what)
{
    if (m) m->err = what;
    return code;
}

// The pinned buffer's layout for a batch of B: byte offsets of its parts.
struct Stage {
    size_t x, cls, reg, loss, y, prob, ent, end;
    size_t ex, em, ep, eh, ec, er;   // an ensemble's call: rows, mean and std, its answers
    Stage(int B, int n_in, int n_out)
    {
        size_t o = 0;
        auto part = [&](size_t words) {
            const size_t at = o;
            o += (4 * words + 255) / 256 * 256;
            return at;
        };
        const size_t b = (size_t)B;
        x = part(b * n_in);
        cls = part(b);
        reg = part(b * (n_out - NCLS));
        loss = part(b);
        y = part(b * n_out);
        prob = part(b * NCLS);
        ent = part(b);
        end = o;
        // (on its own in the buffer: a call uses either these or those above)
        o = 0;
        ex = part(2 * b * n_in);
        em = part(4 * (size_t)n_in);
        ep = part(2 * b * NCLS);
        eh = part(2 * b);
        ec = part(b);
        er = part(b * (n_out - NCLS));
        end = std::max(end, o);
    }
};

template <bool TA, bool TB>
void gemm(hipStream_t st, int M, int N, int K, const bf16* A, int lda, const bf16* B, int ldb, float* C, int ldc,
          bf16* Cb, int ldcb, const float* bias, bool relu, const float* csrc = nullptr, int ldcs = 0,
          float* csum = nullptr)
{
    const dim3 grid((N + GN - 1) / GN, (M + GM - 1) / GM);
    k_gemm<TA, TB><<<grid, 256, 0, st>>>(M, N, K, A, lda, B, ldb, C, ldc, Cb, ldcb, bias, relu ? 1 : 0, csrc, ldcs,
                                         csum);
}

void free_mlp(sl_mlp* m)
{
    if (m->pool) (void)hipFree(m->pool);
    if (m->stage) (void)hipHostFree(m->stage);
    for (hipEvent_t e : m->half)
        if (e) (void)hipEventDestroy(e);
    if (m->stream) (void)hipStreamDestroy(m->stream);
}

// Device memory of the model: called once to measure (base NULL) and once to place.
size_t place(sl_mlp* m, char* base)
{
    size_t o = 0;
    auto part = [&](auto*& p, size_t count) {
        using T = std::remove_reference_t<decltype(*p)>;
        p = reinterpret_cast<T*>(base + o);
        o += (count * sizeof(T) + 255) / 256 * 256;
    };
    auto flat = [&](float*& start, auto W, auto b) {
        start = reinterpret_cast<float*>(base + o);
        const size_t o0 = o;
        for (Layer& L : m->L) {
            part(L.*W, (size_t)L.ldin * L.ldout);
            part(L.*b, L.ldout);
        }
        m->n_flat = (o - o0) / sizeof(float);
    };
    flat(m->params, &Layer::W, &Layer::b);
    flat(m->grads, &Layer::gW, &Layer::gb);
    float* second = nullptr;
    flat(m->moments, &Layer::mW, &Layer::mb);
    flat(second, &Layer::vW, &Layer::vb);
    const size_t mb = (size_t)m->max_batch;
    for (int k = 0; k < NL; k++) {
        Layer& L = m->L[k];
        const size_t na = mb * L.ldout;
        part(m->dZ[k], na);
        if (m->chain) {
            part(L.Wf, (size_t)32 * k_steps(L.ldin) * L.ldout);
            part(L.Wr, (size_t)32 * k_steps(L.ldout) * L.ldin);
            part(m->Ht[k], (size_t)L.ldin * m->ldb);
            part(m->dZt[k], (size_t)L.ldout * m->ldb);
        } else {
            part(L.Wb, (size_t)L.ldin * L.ldout);
            part(m->Z[k], na);
            part(m->Hb[k], na);
            part(m->dZb[k], na);
        }
    }
    part(m->xin, mb * m->n_in);
    part(m->prob, mb * NCLS);
    part(m->ent, mb);
    if (m->chain) {
        part(m->yout, mb * m->n_out);
    } else {
        part(m->xb, mb * m->L[0].ldin);
        part(m->reg, mb * (m->n_out - NCLS));
        part(m->loss_s, mb);
        part(m->cls, mb);
    }
    return o;
}

// Waits for the net's stream; whether that and the launches before it went well.
bool finished(const sl_mlp* m)
{
    const bool launched = hipGetLastError() == hipSuccess;
    return hipStreamSynchronize(m->stream) == hipSuccess && launched;
}

// The padded floats [f0, f1) of the parameters' layout that the caller's unpadded one has too:
// f(padded offset, unpadded offset, count) for each run of them.
template <class F>
void each_run(const sl_mlp* m, size_t f0, size_t f1, F f)
{
    size_t user = 0;
    for (const Layer& L : m->L) {
        auto rows = [&](const float* start, size_t count) {
            const size_t at = start - m->params, ld = L.ldout, len = L.out;
            for (size_t i = f0 > at ? (f0 - at) / ld : 0; i < count && at + i * ld < f1; i++) {
                const size_t lo = std::max(at + i * ld, f0), hi = std::min(at + i * ld + len, f1);
                if (lo < hi) f(lo, user + lo - at - i * (ld - len), hi - lo);
            }
            user += count * len;
        };
        rows(L.W, L.in);
        rows(L.b, 1);
    }
}

// The caller's parameters to the device, padded, with their bfloat16 copies.
int push_params(sl_mlp* m, const float* w)
{
    float* host = reinterpret_cast<float*>(m->stage);
    const size_t per = m->stage_bytes / sizeof(float);
    for (size_t f0 = 0; f0 < m->n_flat; f0 += per) {
        const size_t n = std::min(per, m->n_flat - f0);
        std::memset(host, 0, sizeof(float) * n);
        each_run(m, f0, f0 + n, [&](size_t at, size_t user, size_t c) { std::memcpy(host + (at - f0), w + user, sizeof(float) * c); });
        if (hipMemcpyAsync(m->params + f0, host, sizeof(float) * n, hipMemcpyHostToDevice, m->stream) != hipSuccess ||
            (f0 + n < m->n_flat && hipStreamSynchronize(m->stream) != hipSuccess))
            return SL_E_HIP;
    }
    for (Layer& L : m->L) {
        const int nw = L.ldin * L.ldout;
        k_weights_bf16<<<(nw + 255) / 256, 256, 0, m->stream>>>(L.ldin, L.ldout, L.W, L.Wb, L.Wf, L.Wr);
    }
    const bool ok = hipMemsetAsync(m->moments, 0, 2 * sizeof(float) * m->n_flat, m->stream) == hipSuccess;
    if (!finished(m) || !ok) return SL_E_HIP;
    m->t = 0;
    return SL_OK;
}

// A flat device block (parameters or gradients) into the caller's unpadded layout.
int pull_flat(sl_mlp* m, const float* dev, float* out)
{
    const float* host = reinterpret_cast<const float*>(m->stage);
    const size_t per = m->stage_bytes / sizeof(float);
    for (size_t f0 = 0; f0 < m->n_flat; f0 += per) {
        const size_t n = std::min(per, m->n_flat - f0);
        if (hipMemcpyAsync(m->stage, dev + f0, sizeof(float) * n, hipMemcpyDeviceToHost, m->stream) != hipSuccess ||
            hipStreamSynchronize(m->stream) != hipSuccess)
            return SL_E_HIP;
        each_run(m, f0, f0 + n, [&](size_t at, size_t user, size_t c) { std::memcpy(out + user, host + (at - f0), sizeof(float) * c); });
    }
    return SL_OK;
}

// ---- chain form ------------------------------------------------------------------------

ChainArgs chain_args(sl_mlp* const* ms, int n, int B, bool one_input)
{
    ChainArgs a{};
    sl_mlp* m = ms[0];
    for (int j = 0; j < n; j++) {
        a.at[j].pool = ms[j]->pool - m->pool;
        a.at[j].stage = ms[j]->stage_dev - m->stage_dev;
        a.at[j].x = one_input ? 0 : a.at[j].stage;
    }
    const Stage s(m->max_batch, m->n_in, m->n_out);
    auto at = [&](size_t o) { return reinterpret_cast<float*>(m->stage_dev + o); };
    a.B = B;
    a.n_in = m->n_in;
    a.n_out = m->n_out;
    a.ld[0] = m->L[0].ldin;
    for (int k = 0; k < NL; k++) {
        const Layer& L = m->L[k];
        a.ld[k + 1] = L.ldout;
        a.Wf[k] = L.Wf;
        a.Wr[k] = L.Wr;
        a.b[k] = L.b;
        a.Ht[k] = m->Ht[k];
        a.dZt[k] = m->dZt[k];
        a.dZ[k] = m->dZ[k];
    }
    a.ldb = m->ldb;
    a.x = at(s.x);
    a.cls = reinterpret_cast<int*>(m->stage_dev + s.cls);
    a.reg = at(s.reg);
    a.loss = at(s.loss);
    a.y = at(s.y);
    a.prob = at(s.prob);
    a.ent = at(s.ent);
    return a;
}

// A batch of B of each of ms[0 .. n - 1] (alike, n <= MEMBERS), on the first one's stream;
// inference reads the first one's input rows.
template <bool TRAIN>
void launch_chain(sl_mlp* const* ms, int n, int B, const ChainArgs& a)
{
    const sl_mlp* m = ms[0];
    int widest = 0;   // column tiles of the widest layer: one wavefront each, up to CHAIN_WAVES
    for (const Layer& L : m->L) widest = std::max(widest, L.ldout / 16);
    const int threads = 64 * std::min(widest, CHAIN_WAVES);
    const dim3 grid((B + CHAIN_ROWS - 1) / CHAIN_ROWS, n);
    const bool f0 = m->L[0].ldin > 32, fl = m->L[NL - 1].ldout > 32;
    if (f0)
        fl ? k_chain<TRAIN, KF, KF><<<grid, threads, 0, m->stream>>>(a) : k_chain<TRAIN, KF, 1><<<grid, threads, 0, m->stream>>>(a);
    else
        fl ? k_chain<TRAIN, 1, KF><<<grid, threads, 0, m->stream>>>(a) : k_chain<TRAIN, 1, 1><<<grid, threads, 0, m->stream>>>(a);
}

template <bool TRAIN>
void launch_chain(sl_mlp* const* ms, int n, int B)
{
    launch_chain<TRAIN>(ms, n, B, chain_args(ms, n, B, !TRAIN));
}

template <bool STEP>
void launch_wgrad(sl_mlp* const* ms, int n, int B, const Adam* adam)
{
    WgradArgs a{};
    sl_mlp* m = ms[0];
    a.B = B;
    a.ldb = m->ldb;
    for (int j = 0; j < n; j++) {
        a.pool[j] = ms[j]->pool - m->pool;
        if (adam) a.adam[j] = adam[j];
    }
    a.ld[0] = m->L[0].ldin;
    int bias = 0;
    for (int k = 0; k < NL; k++) {
        const Layer& L = m->L[k];
        a.ld[k + 1] = L.ldout;
        a.tile0[k + 1] = a.tile0[k] + (L.ldin / 16) * (L.ldout / 16);
        bias += (L.ldout + 31) / 32;
        a.bias0[k + 1] = bias;
        a.Ht[k] = m->Ht[k];
        a.dZt[k] = m->dZt[k];
        a.dZ[k] = m->dZ[k];
        a.W[k] = L.W;
        a.mW[k] = L.mW;
        a.vW[k] = L.vW;
        a.gW[k] = L.gW;
        a.Wf[k] = L.Wf;
        a.Wr[k] = L.Wr;
        a.b[k] = L.b;
        a.mb[k] = L.mb;
        a.vb[k] = L.vb;
        a.gb[k] = L.gb;
    }
    a.wblocks = (a.tile0[NL] + 3) / 4;
    k_wgrad<STEP><<<dim3(a.wblocks + bias, n), 256, 0, m->stream>>>(a);
}

// ---- layer form ------------------------------------------------------------------------

// Forward pass of a batch already packed into m->xb: hidden layers keep their
// post-activation values (binary32 in Z, whose sign is also the ReLU mask, and
// bfloat16 in Hb for the next product); the last layer's outputs are in Z[NL-1].
void forward(sl_mlp* m, int B)
{
    const bf16* in = m->xb;
    for (int k = 0; k < NL; k++) {
        Layer& L = m->L[k];
        const bool last = k == NL - 1;
        gemm<false, false>(m->stream, B, L.ldout, L.ldin, in, L.ldin, L.Wb, L.ldout, m->Z[k], L.ldout,
                           last ? nullptr : m->Hb[k], L.ldout, L.b, !last);
        in = m->Hb[k];
    }
}

// Backward pass after forward() and the loss kernel (dZ[NL-1] set): parameter
// gradients into gW, gb.
void backward(sl_mlp* m, int B)
{
    for (int k = NL - 1; k >= 0; k--) {
        Layer& L = m->L[k];
        const bf16* Hprev = k ? m->Hb[k - 1] : m->xb;
        // weight gradient H^T dZ, and the bias gradient (column sums of dZ) in the same launch
        gemm<true, false>(m->stream, L.ldin, L.ldout, B, Hprev, L.ldin, m->dZb[k], L.ldout, L.gW, L.ldout, nullptr, 0,
                          nullptr, false, m->dZ[k], L.ldout, L.gb);
        if (k > 0) {
            gemm<false, true>(m->stream, B, L.ldin, L.ldout, m->dZb[k], L.ldout, L.Wb, L.ldout, m->dZ[k - 1], L.ldin,
                              nullptr, 0, nullptr, false);
            const int n = B * L.ldin;
            k_relu_back<<<(n + 255) / 256, 256, 0, m->stream>>>(n, m->Z[k - 1], m->dZ[k - 1], m->dZb[k - 1]);
        }
    }
}

int load_batch(sl_mlp* m, int B, const float* x)
{
    if (hipMemcpyAsync(m->xin, x, 4 * (size_t)B * m->n_in, hipMemcpyHostToDevice, m->stream) != hipSuccess)
        return SL_E_HIP;
    const int ld0 = m->L[0].ldin, n = B * ld0;
    k_pack_input<<<(n + 255) / 256, 256, 0, m->stream>>>(B, m->n_in, ld0, m->xin, m->xb);
    return hipGetLastError() == hipSuccess ? SL_OK : SL_E_HIP;
}

// ---- both forms --------------------------------------------------------------------------

float mean_loss(const float* ls, int B)
{
    double sum = 0;
    for (int b = 0; b < B; b++) sum += ls[b];
    return (float)(sum / B);
}

Adam adam_step(const sl_mlp* m, float lr)
{
    const float b1 = 0.9f, b2 = 0.999f;
    const long long t = m->t + 1;
    return Adam{lr, b1, b2, 1e-8f, 1.f - std::pow(b1, (float)t), 1.f - std::pow(b2, (float)t)};
}

// Whether one launch can carry them all: different nets in the chain form, laid out alike on
// one device.
bool alike(sl_mlp* const* ms, int n)
{
    auto kind = [](const sl_mlp& m) { return sl::NetKind{m.device, m.chain, m.n_in, m.width, m.n_out, m.max_batch}; };
    for (int j = 0; j < n; j++) {
        if (!sl::shares_launch(kind(*ms[0]), kind(*ms[j]))) return false;
        for (int i = 0; i < j; i++)
            if (ms[i] == ms[j]) return false;
    }
    return true;
}

// Forward, loss, backward and, with adam, the update of a labelled batch; the mean loss (of
// the parameters before the update) to *loss.
int train_pass(sl_mlp* m, int B, const float* x, const int* cls, const float* reg, float* loss, const Adam* adam)
{
    for (int b = 0; b < B; b++)
        if (cls[b] < 0 || cls[b] >= NCLS) return mlp_err(m, SL_E_ARG, "class label outside 0..2");
    const int nr = m->n_out - NCLS;
    const Stage s(m->max_batch, m->n_in, m->n_out);
    const float* ls = reinterpret_cast<const float*>(m->stage + (m->chain ? s.loss : 0));
    if (m->chain) {
        std::memcpy(m->stage + s.x, x, 4 * (size_t)B * m->n_in);
        std::memcpy(m->stage + s.cls, cls, 4 * (size_t)B);
        std::memcpy(m->stage + s.reg, reg, 4 * (size_t)B * nr);
        launch_chain<true>(&m, 1, B);
        adam ? launch_wgrad<true>(&m, 1, B, adam) : launch_wgrad<false>(&m, 1, B, nullptr);
    } else {
        if (load_batch(m, B, x)) return mlp_err(m, SL_E_HIP, "input upload failed");
        if (hipMemcpyAsync(m->cls, cls, 4 * (size_t)B, hipMemcpyHostToDevice, m->stream) != hipSuccess ||
            hipMemcpyAsync(m->reg, reg, 4 * (size_t)B * nr, hipMemcpyHostToDevice, m->stream) != hipSuccess)
            return mlp_err(m, SL_E_HIP, "label upload failed");
        forward(m, B);
        const Layer& L = m->L[NL - 1];
        k_loss<<<(B + 255) / 256, 256, 0, m->stream>>>(B, m->n_out, L.ldout, m->Z[NL - 1], m->cls, m->reg,
                                                       m->dZ[NL - 1], m->dZb[NL - 1], m->loss_s);
        if (hipMemcpyAsync(m->stage, m->loss_s, 4 * (size_t)B, hipMemcpyDeviceToHost, m->stream) != hipSuccess)
            return mlp_err(m, SL_E_HIP, "loss read-back failed");
        backward(m, B);
        if (adam)
            for (Layer& Lk : m->L) {
                const int nw = Lk.ldin * Lk.ldout;
                k_adam<<<(nw + 255) / 256, 256, 0, m->stream>>>(nw, Lk.W, Lk.Wb, Lk.gW, Lk.mW, Lk.vW, *adam);
                k_adam<<<(Lk.ldout + 255) / 256, 256, 0, m->stream>>>(Lk.ldout, Lk.b, nullptr, Lk.gb, Lk.mb, Lk.vb,
                                                                      *adam);
            }
    }
    if (!finished(m)) return mlp_err(m, SL_E_HIP, "training pass failed");
    if (loss) *loss = mean_loss(ls, B);
    return SL_OK;
}

int check_batch(sl_mlp* m, int B, const void* x)
{
    if (!m) return SL_E_ARG;
    if (B < 1 || B > m->max_batch || !x) return mlp_err(m, SL_E_ARG, "batch size outside [1, max_batch] or NULL input");
    return SL_OK;
}

// sl_mlp_ensemble, the rows and their normalising in T.
template <class T>
int ensemble(sl_mlp* const* ms, int n, long long rows, const T* x, const T* mean, const T* std, int* cls, float* reg,
             double* prob, double* ent)
{
    if (!ms || n < 1 || rows < 0) return SL_E_ARG;
    for (int j = 0; j < n; j++)
        if (!ms[j]) return SL_E_ARG;
    sl_mlp* m = ms[0];
    if (!mean || !std || (rows > 0 && !(x && cls && reg && prob && ent))) return mlp_err(m, SL_E_ARG, "an array is NULL");
    if (n > MEMBERS || !alike(ms, n)) return mlp_err(m, SL_E_STATE, "the nets cannot share launches");
    const int n_in = m->n_in, nr = m->n_out - NCLS;
    // two batches in flight, each in its half of the buffers: one is copied in and the other's
    // answers out while the device works
    const int per = std::max(1, m->max_batch / 2);
    const Stage s(m->max_batch, n_in, m->n_out);
    std::memcpy(m->stage + s.em, mean, sizeof(T) * n_in);
    std::memcpy(m->stage + s.em + sizeof(T) * n_in, std, sizeof(T) * n_in);
    const bool halves = m->max_batch > 1;
    auto at = [&](char* base, size_t part, size_t bytes, long long k) { return base + part + (halves && k % 2 ? bytes * per : 0); };
    auto size = [&](long long k) { return (int)std::min<long long>(per, rows - k * per); };
    auto collect = [&](long long k) -> int {
        if (hipEventSynchronize(m->half[k % 2]) != hipSuccess) return mlp_err(m, SL_E_HIP, "ensemble pass failed");
        const size_t b0 = (size_t)k * per, B = size(k);
        std::memcpy(prob + NCLS * b0, at(m->stage, s.ep, 8 * NCLS, k), 8 * NCLS * B);
        std::memcpy(ent + b0, at(m->stage, s.eh, 8, k), 8 * B);
        std::memcpy(cls + b0, at(m->stage, s.ec, 4, k), 4 * B);
        std::memcpy(reg + nr * b0, at(m->stage, s.er, 4 * (size_t)nr, k), 4 * nr * B);
        return SL_OK;
    };
    auto issue = [&](long long k) -> int {
        const int B = size(k);
        std::memcpy(at(m->stage, s.ex, sizeof(T) * n_in, k), x + (size_t)k * per * n_in, sizeof(T) * B * n_in);
        auto dev = [&](size_t part, size_t bytes) { return at(m->stage_dev, part, bytes, k); };
        const T* em = reinterpret_cast<const T*>(m->stage_dev + s.em);
        k_normalise<<<(B * n_in + 255) / 256, 256, 0, m->stream>>>(
            B, n_in, reinterpret_cast<const T*>(dev(s.ex, sizeof(T) * n_in)), em, em + n_in, m->xin);
        ChainArgs c = chain_args(ms, n, B, true);
        EnsembleArgs e{};
        for (int j = 0; j < n; j++) c.at[j].stage = e.at[j] = c.at[j].pool;
        c.x = m->xin;
        c.y = m->yout;
        c.prob = m->prob;
        c.ent = m->ent;
        launch_chain<false>(ms, n, B, c);
        e.n = n;
        e.B = B;
        e.n_out = m->n_out;
        e.y = m->yout;
        e.prob = m->prob;
        e.cls = reinterpret_cast<int*>(dev(s.ec, 4));
        e.reg = reinterpret_cast<float*>(dev(s.er, 4 * (size_t)nr));
        e.p = reinterpret_cast<double*>(dev(s.ep, 8 * NCLS));
        e.ent = reinterpret_cast<double*>(dev(s.eh, 8));
        k_ensemble<<<(B + 63) / 64, 64, 0, m->stream>>>(e);
        if (hipGetLastError() != hipSuccess || hipEventRecord(m->half[k % 2], m->stream) != hipSuccess)
            return mlp_err(m, SL_E_HIP, "ensemble pass failed");
        return SL_OK;
    };
    return sl::run_ahead((rows + per - 1) / per, halves ? 2 : 1, issue, collect, [&] { (void)hipStreamSynchronize(m->stream); });
}

}  // namespace

extern "C" {

int sl_mlp_create(sl_mlp** out, int n_in, int width, int n_out, int max_batch, unsigned long long seed)
{
    if (!out) return SL_E_ARG;
    *out = nullptr;
    if (n_in < 1 || width < 16 || n_out <= NCLS || max_batch < 1 || n_in > 4096 || width > 4096 || n_out > 4096)
        return SL_E_ARG;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return SL_E_NOGPU;
    sl_mlp* m = new (std::nothrow) sl_mlp();
    if (!m) return SL_E_ARG;
    m->n_in = n_in;
    m->width = width;
    m->n_out = n_out;
    m->max_batch = max_batch;
    m->ldb = (max_batch + 31) / 32 * 32;
    const int dims[NL + 1] = {n_in, width, width, width, n_out};
    m->chain = true;
    for (int k = 0; k < NL; k++) {
        Layer& L = m->L[k];
        L.in = dims[k];
        L.out = dims[k + 1];
        L.ldin = pad16(L.in);
        L.ldout = pad16(L.out);
        if (L.ldin > CHAIN_MAX || L.ldout > CHAIN_MAX) m->chain = false;
    }
    auto fail = [&](int code) {
        free_mlp(m);
        delete m;
        return code;
    };
    if (hipGetDevice(&m->device) != hipSuccess ||
        hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) != hipSuccess)
        return fail(SL_E_HIP);
    for (hipEvent_t& e : m->half)
        if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return fail(SL_E_HIP);
    if (hipMalloc(&m->pool, place(m, nullptr)) != hipSuccess) return fail(SL_E_HIP);
    place(m, m->pool);
    // the fragments' parts past a layer's widths are zeros for good
    if (m->chain)
        for (Layer& L : m->L)
            if (hipMemsetAsync(L.Wf, 0, 2 * (size_t)32 * k_steps(L.ldin) * L.ldout, m->stream) != hipSuccess ||
                hipMemsetAsync(L.Wr, 0, 2 * (size_t)32 * k_steps(L.ldout) * L.ldin, m->stream) != hipSuccess)
                return fail(SL_E_HIP);
    m->stage_bytes = sl::pinned_bytes(m->chain, Stage(max_batch, n_in, n_out).end, sizeof(float) * m->n_flat, max_batch);
    if (hipHostMalloc(&m->stage, m->stage_bytes, 0) != hipSuccess ||
        hipHostGetDevicePointer(reinterpret_cast<void**>(&m->stage_dev), m->stage, 0) != hipSuccess)
        return fail(SL_E_HIP);
    // He-uniform initialisation from a SplitMix64 stream
    uint64_t s = seed;
    auto rnd = [&]() {
        uint64_t z = (s += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        z ^= z >> 31;
        return ((z >> 11) + 0.5) * (1.0 / 9007199254740992.0);
    };
    float* w = new (std::nothrow) float[sl_mlp_n_params(m)], *next = w;
    if (!w) return fail(SL_E_STATE);
    for (const Layer& L : m->L) {
        const double lim = std::sqrt(6.0 / L.in);
        for (int e = 0; e < L.in * L.out; e++) *next++ = (float)((2 * rnd() - 1) * lim);
        for (int e = 0; e < L.out; e++) *next++ = 0.f;
    }
    const int rc = push_params(m, w);
    delete[] w;
    if (rc) return fail(SL_E_HIP);
    *out = m;
    return SL_OK;
}

int sl_mlp_device(const sl_mlp* m) { return m ? m->device : SL_E_ARG; }

int sl_mlp_n_params(const sl_mlp* m)
{
    if (!m) return SL_E_ARG;
    int n = 0;
    for (const Layer& L : m->L) n += L.in * L.out + L.out;
    return n;
}

// Flat parameter layout: for each layer W[in][out] (row-major) then b[out].
int sl_mlp_get_params(sl_mlp* m, float* w)
{
    if (!m || !w) return SL_E_ARG;
    if (pull_flat(m, m->params, w)) return mlp_err(m, SL_E_HIP, "parameter read-back failed");
    return SL_OK;
}

int sl_mlp_set_params(sl_mlp* m, const float* w)
{
    if (!m || !w) return SL_E_ARG;
    if (push_params(m, w)) return mlp_err(m, SL_E_HIP, "parameter upload failed");
    return SL_OK;
}

int sl_mlp_forward(sl_mlp* m, int B, const float* x, float* y, float* prob, float* ent)
{
    int rc = check_batch(m, B, x);
    if (rc) return rc;
    if (m->chain) {
        const Stage s(m->max_batch, m->n_in, m->n_out);
        std::memcpy(m->stage + s.x, x, 4 * (size_t)B * m->n_in);
        launch_chain<false>(&m, 1, B);
        if (!finished(m)) return mlp_err(m, SL_E_HIP, "forward failed");
        if (y) std::memcpy(y, m->stage + s.y, 4 * (size_t)B * m->n_out);
        if (prob) std::memcpy(prob, m->stage + s.prob, 4 * (size_t)B * NCLS);
        if (ent) std::memcpy(ent, m->stage + s.ent, 4 * (size_t)B);
        return SL_OK;
    }
    if (load_batch(m, B, x)) return mlp_err(m, SL_E_HIP, "input upload failed");
    forward(m, B);
    const Layer& L = m->L[NL - 1];
    k_predict<<<(B + 255) / 256, 256, 0, m->stream>>>(B, L.ldout, m->Z[NL - 1], m->prob, m->ent);
    if (prob && hipMemcpyAsync(prob, m->prob, 4 * (size_t)B * NCLS, hipMemcpyDeviceToHost, m->stream) != hipSuccess)
        return mlp_err(m, SL_E_HIP, "probability read-back failed");
    if (ent && hipMemcpyAsync(ent, m->ent, 4 * (size_t)B, hipMemcpyDeviceToHost, m->stream) != hipSuccess)
        return mlp_err(m, SL_E_HIP, "entropy read-back failed");
    if (!finished(m)) return mlp_err(m, SL_E_HIP, "forward failed");
    // the outputs through the pinned buffer, whole padded rows at a time
    const int per = (int)std::min<size_t>(B, m->stage_bytes / (4 * (size_t)L.ldout));
    for (int b0 = 0; y && b0 < B; b0 += per) {
        const int n = std::min(per, B - b0);
        if (hipMemcpyAsync(m->stage, m->Z[NL - 1] + (size_t)b0 * L.ldout, 4 * (size_t)n * L.ldout, hipMemcpyDeviceToHost, m->stream) !=
                hipSuccess ||
            hipStreamSynchronize(m->stream) != hipSuccess)
            return mlp_err(m, SL_E_HIP, "output read-back failed");
        for (int b = 0; b < n; b++)
            std::memcpy(y + (size_t)(b0 + b) * m->n_out, m->stage + 4 * (size_t)b * L.ldout, 4 * (size_t)m->n_out);
    }
    return SL_OK;
}

int sl_mlp_ensemble(sl_mlp* const* ms, int n, long long rows, const double* x, const double* mean, const double* std, int* cls,
                    float* reg, double* prob, double* ent)
{
    return ensemble(ms, n, rows, x, mean, std, cls, reg, prob, ent);
}

int sl_mlp_ensemble32(sl_mlp* const* ms, int n, long long rows, const float* x, const float* mean, const float* std, int* cls,
                      float* reg, double* prob, double* ent)
{
    return ensemble(ms, n, rows, x, mean, std, cls, reg, prob, ent);
}

int sl_mlp_gradients(sl_mlp* m, int B, const float* x, const int* cls, const float* reg, float* loss, float* grads)
{
    int rc = check_batch(m, B, x);
    if (rc) return rc;
    if (!cls || !reg) return mlp_err(m, SL_E_ARG, "labels are NULL");
    rc = train_pass(m, B, x, cls, reg, loss, nullptr);
    if (rc) return rc;
    if (grads && pull_flat(m, m->grads, grads)) return mlp_err(m, SL_E_HIP, "gradient read-back failed");
    return SL_OK;
}

int sl_mlp_train_step(sl_mlp* m, int B, const float* x, const int* cls, const float* reg, float lr, float* loss)
{
    int rc = check_batch(m, B, x);
    if (rc) return rc;
    if (!cls || !reg || !(lr > 0)) return mlp_err(m, SL_E_ARG, "labels are NULL or lr <= 0");
    const Adam adam = adam_step(m, lr);
    rc = train_pass(m, B, x, cls, reg, loss, &adam);
    if (rc) return rc;
    m->t++;
    return SL_OK;
}

int sl_mlp_train_rows(sl_mlp* const* ms, int n, int B, int batches, long long n_rows, const float* x, const int* cls,
                      const float* reg, const long long* idx, float lr, float* loss)
{
    if (!ms || n < 1 || batches < 0) return SL_E_ARG;
    for (int j = 0; j < n; j++) {
        const int rc = check_batch(ms[j], B, x);
        if (rc) return rc;
        if (!cls || !reg || !idx || !(lr > 0)) return mlp_err(ms[j], SL_E_ARG, "labels or rows are NULL or lr <= 0");
        if (ms[j]->n_in != ms[0]->n_in || ms[j]->n_out != ms[0]->n_out)
            return mlp_err(ms[j], SL_E_ARG, "nets of one ensemble have the same inputs and outputs");
    }
    auto at = [&](long long k, int j) { return idx + ((size_t)k * n + j) * B; };   // rows of batch k of net j
    for (size_t e = 0; e < (size_t)batches * n * B; e++) {
        sl_mlp* m = ms[e / B % n];
        if (idx[e] < 0 || idx[e] >= n_rows) return mlp_err(m, SL_E_ARG, "row index outside the data");
        if (cls[idx[e]] < 0 || cls[idx[e]] >= NCLS) return mlp_err(m, SL_E_ARG, "class label outside 0..2");
    }
    const int n_in = ms[0]->n_in, nr = ms[0]->n_out - NCLS;
    auto rows = [&](const long long* r, float* px, int* pc, float* pr) {
        for (int b = 0; b < B; b++) {
            std::memcpy(px + (size_t)b * n_in, x + r[b] * n_in, 4 * (size_t)n_in);
            pc[b] = cls[r[b]];
            std::memcpy(pr + (size_t)b * nr, reg + r[b] * nr, 4 * (size_t)nr);
        }
    };
    if (!alike(ms, n)) {
        const size_t words = (size_t)B * (n_in + 1 + nr);
        float* buf = new (std::nothrow) float[words];
        if (!buf) return mlp_err(ms[0], SL_E_STATE, "out of memory");
        float* pr = buf + (size_t)B * n_in;
        int* pc = reinterpret_cast<int*>(pr + (size_t)B * nr);
        int rc = SL_OK;
        for (int k = 0; k < batches && rc == SL_OK; k++)
            for (int j = 0; j < n && rc == SL_OK; j++) {
                rows(at(k, j), buf, pc, pr);
                rc = sl_mlp_train_step(ms[j], B, buf, pc, pr, lr, loss ? loss + (size_t)k * n + j : nullptr);
                if (rc && j) ms[0]->err = ms[j]->err;
            }
        delete[] buf;
        return rc;
    }
    // Batches that take up to half of the pinned buffer are gathered into its halves in turn,
    // one while the device trains on the other.
    const Stage s(ms[0]->max_batch, n_in, nr + NCLS);
    const int ahead = 2 * B <= ms[0]->max_batch ? 2 : 1;
    const size_t half = ahead == 2 ? (size_t)(ms[0]->max_batch / 2) : 0;   // rows
    for (int j0 = 0; j0 < n; j0 += MEMBERS) {
        const int g = std::min(n - j0, MEMBERS);
        sl_mlp* const* mg = ms + j0;
        auto part = [&](sl_mlp* m, size_t p, size_t bytes, long long k) { return m->stage + p + k % ahead * half * bytes; };
        auto collect = [&](long long k) -> int {
            if (hipEventSynchronize(mg[0]->half[k % 2]) != hipSuccess) return mlp_err(ms[0], SL_E_HIP, "training pass failed");
            for (int j = 0; loss && j < g; j++)
                loss[(size_t)k * n + j0 + j] = mean_loss(reinterpret_cast<const float*>(part(mg[j], s.loss, 4, k)), B);
            return SL_OK;
        };
        ChainArgs c = chain_args(mg, g, B, false);
        const ChainArgs c0 = c;
        auto issue = [&](long long k) -> int {
            Adam adam[MEMBERS];
            for (int j = 0; j < g; j++) {
                sl_mlp* m = mg[j];
                adam[j] = adam_step(m, lr);
                rows(at(k, j0 + j), reinterpret_cast<float*>(part(m, s.x, 4 * (size_t)n_in, k)),
                     reinterpret_cast<int*>(part(m, s.cls, 4, k)), reinterpret_cast<float*>(part(m, s.reg, 4 * (size_t)nr, k)));
            }
            const size_t r0 = k % ahead * half;
            c.x = c0.x + r0 * n_in;
            c.cls = c0.cls + r0;
            c.reg = c0.reg + r0 * nr;
            c.loss = c0.loss + r0;
            launch_chain<true>(mg, g, B, c);
            launch_wgrad<true>(mg, g, B, adam);
            if (hipGetLastError() != hipSuccess || hipEventRecord(mg[0]->half[k % 2], mg[0]->stream) != hipSuccess)
                return mlp_err(ms[0], SL_E_HIP, "training pass failed");
            for (int j = 0; j < g; j++) mg[j]->t++;   // a step that was sent
            return SL_OK;
        };
        if (const int rc = sl::run_ahead(batches, ahead, issue, collect, [&] { (void)hipStreamSynchronize(mg[0]->stream); })) return rc;
    }
    return SL_OK;
}

int sl_mlp_forward_all(sl_mlp* const* ms, int n, int B, const float* x, float* y, float* prob, float* ent)
{
    if (!ms || n < 1) return SL_E_ARG;
    for (int j = 0; j < n; j++) {
        const int rc = check_batch(ms[j], B, x);
        if (rc) return rc;
        if (ms[j]->n_in != ms[0]->n_in || ms[j]->n_out != ms[0]->n_out)
            return mlp_err(ms[j], SL_E_ARG, "nets of one ensemble have the same inputs and outputs");
    }
    const size_t ny = (size_t)B * ms[0]->n_out, np = (size_t)B * NCLS;
    const bool together = alike(ms, n);
    const Stage s(ms[0]->max_batch, ms[0]->n_in, ms[0]->n_out);
    for (int j0 = 0; j0 < n; j0 += MEMBERS) {
        const int k = std::min(n - j0, MEMBERS);
        if (together) {
            std::memcpy(ms[j0]->stage + s.x, x, 4 * (size_t)B * ms[0]->n_in);
            launch_chain<false>(ms + j0, k, B);
            if (!finished(ms[j0])) return mlp_err(ms[0], SL_E_HIP, "forward failed");
        }
        for (int j = j0; j < j0 + k; j++) {
            float *yj = y ? y + j * ny : nullptr, *pj = prob ? prob + j * np : nullptr, *ej = ent ? ent + (size_t)j * B : nullptr;
            if (together) {
                if (yj) std::memcpy(yj, ms[j]->stage + s.y, 4 * ny);
                if (pj) std::memcpy(pj, ms[j]->stage + s.prob, 4 * np);
                if (ej) std::memcpy(ej, ms[j]->stage + s.ent, 4 * (size_t)B);
            } else if (const int rc = sl_mlp_forward(ms[j], B, x, yj, pj, ej)) {
                if (j) ms[0]->err = ms[j]->err;
                return rc;
            }
        }
    }
    return SL_OK;
}

const char* sl_mlp_last_error(const sl_mlp* m) { return m ? m->err.c_str() : "NULL model"; }

void sl_mlp_destroy(sl_mlp* m)
{
    if (!m) return;
    if (m->stream) (void)hipStreamSynchronize(m->stream);
    free_mlp(m);
    delete m;
}

}  // extern "C"
