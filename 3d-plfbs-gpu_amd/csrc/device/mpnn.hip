// Warm-start message-passing network on the cell graph (gfx950).
//
// 6 layers, hidden width 64, every MLP Linear -> SiLU -> Linear:
//   h  = enc(x)                                  x: [N,16] node inputs
//   repeat 6: m_e = msg([h[dst_e], h[src_e], f_e])    f_e: [E,16] edge inputs
//             a_t = sum_{dst_e = t} m_e / max(deg_t, 1)
//             h   = h + upd([h, a])
//   y  = dec(h)                                  y: [N,16]
// Directed edges are sorted by (dst, src); aggregation and every backward
// scatter walk fixed per-node edge lists, so no float atomics are used and
// results are bitwise reproducible.
//
// A layer is one kernel forward (k_layer_fwd) and three backward (k_node_bwd for the
// update MLP, k_msg_bwd for the message MLP, k_dh_out for the edges' source side).  A
// block walks over tiles of consecutive nodes with at most kTileNodes nodes and, if
// the tile has more than one node, kTileRows in-edges; the edge rows [h_dst, h_src, f],
// hidden activations and messages of a tile live in LDS only, so neither the E x 144
// inputs nor the E x 64 activations and messages pass through memory.  The backward
// pass computes the hidden activations again from the bfloat16 node states instead
// of keeping them.
//
// Every product runs on the matrix cores as v_mfma_f32_16x16x16_bf16 with FP32
// accumulation over k in steps of 16; operands are rounded to bfloat16 (nearest even)
// from FP32 activations and master weights.  The node states are kept twice, in
// FP32 for the residual sum and rounded once to bfloat16 as the operand that every
// product uses.  Weights are held as register fragments by the wavefronts, each of
// which owns 16 hidden units.  Weight gradients accumulate in registers over a
// block's tiles; the blocks' FP32 partials are added in a fixed order.  Adam keeps
// FP32 master weights and moments.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstring>
#include <numeric>
#include <vector>

#include "ctx.hpp"
#include "plbfs_mpnn.h"

namespace {

constexpr int kH = 64;           // hidden width
constexpr int kDin = 16;         // node input width (padded)
constexpr int kDedge = 16;       // edge input width (padded)
constexpr int kDout = 16;        // output width (padded)
constexpr int kLayers = 6;
constexpr int kKmsg = 2 * kH + kDedge;  // 144
constexpr int kKupd = 2 * kH;           // 128
constexpr int kMlps = 2 + 2 * kLayers;  // enc, (msg, upd) x 6, dec
constexpr int kT = 256;                 // threads per block

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__host__ __device__ __forceinline__ unsigned short to_bf16(float f) {
    // round to nearest even (inputs are finite)
    unsigned int u = __builtin_bit_cast(unsigned int, f);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}

// SiLU and its derivative: 1 + e^-a from the exponential of the nearest power of two
// and the rest, the argument times log2 e in two parts (Cody and Waite, "Software Manual
// for the Elementary Functions", 1980; log2 e = hi + lo), and the quotients by
// reciprocal and one correction with the remainder that fma gives exactly (Markstein,
// IBM J. Res. Dev. 34, 1990).  expf and the division spend a third of their
// instructions on ranges that do not occur here: a below -88 is taken as -88 (SiLU
// -5e-37 there and 0 below).  NaN stays NaN, and a / (1 + e^-a) at infinity is what it
// is by division: SiLU(inf) = inf, SiLU(-inf) and both derivatives NaN.
// Against 64 bits over [-85, 88] the errors are those of a / (1 + expf(-a)) (largest
// 3.09, mean 0.27668, in 2^-24 of the result), and so are the network's outputs, bit
// for bit.
__device__ __forceinline__ float floor88(float a) { return a < -88.f ? fmaf(a, 0.f, -88.f) : a; }
__device__ __forceinline__ float one_plus_exp(float a) {
#pragma clang fp contract(off)
    const float x = -fminf(a, 88.f);
    const float hi = 1.44269502f, lo = 1.92596299e-8f;
    const float t = x * hi, n = rintf(t);
    const float f = (t - n) + fmaf(x, lo, fmaf(x, hi, -t));
    return 1.0f + ldexpf(__builtin_amdgcn_exp2f(f), (int)n);
}
__device__ __forceinline__ float quot(float a, float d, float r) {  // a / d, r = rcp(d)
    const float q = a * r;
    // (the remainder at q = inf is NaN, which fmaxf drops; it is never below -FLT_MAX)
    return fmaf(fmaxf(fmaf(-q, d, a), -FLT_MAX), r, q);
}
__device__ __forceinline__ float silu(float a) {
    a = floor88(a);
    const float d = one_plus_exp(a);
    return quot(a, d, __builtin_amdgcn_rcpf(d));
}
__device__ __forceinline__ float dsilu(float a) {
    a = floor88(a);
    const float d = one_plus_exp(a), r = __builtin_amdgcn_rcpf(d);
    const float s = fmaf(fmaf(-d, r, 1.0f), r, r);
    return s * (1.0f + a * (1.0f - s));
}

typedef unsigned short u16;

constexpr int kTileRows = 64;   // edges or node rows of a tile
constexpr int kTileNodes = 16;  // nodes of an edge tile
constexpr int kPad = 8;         // bf16 elements behind every row of an LDS tile
constexpr int kMaxParts = 512;  // blocks (weight-gradient partials) of a backward kernel: two a CU

// Nearest even, two values an instruction; equal to to_bf16 for every finite value.
__device__ __forceinline__ bf16x4 pack4(f32x4 v) {
    typedef __bf16 b4 __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(bf16x4, __builtin_convertvector(v, b4));
}

// Operand fragments of the 16x16x16 product D = A B, D(m, n): lane l holds
// A(m = l % 16, k = 4 (l / 16) + q) and B(k = 4 (l / 16) + q, n = l % 16), q = 0..3, and of
// the result D(m = 4 (l / 16) + q, n = l % 16).  With the weights as A and the rows of a
// tile as n, a lane's four results are neighbouring columns of one row.
struct Lane {
    int r, g, w;  // l % 16, l / 16, wavefront
    __device__ __forceinline__ Lane()
        : r(threadIdx.x & 15), g((threadIdx.x & 63) >> 4), w(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) {}
};

__device__ __forceinline__ f32x4 mfma(bf16x4 a, bf16x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// W(k, col) of a row-major weight matrix as the fragment (m = col, k)
__device__ __forceinline__ bf16x4 wfrag(const float *W, int ld, int col, int k) {
    return pack4(f32x4{W[k * ld + col], W[(k + 1) * ld + col], W[(k + 2) * ld + col], W[(k + 3) * ld + col]});
}
// ... its transpose: W(row, k) as the fragment (m = row, k)
__device__ __forceinline__ bf16x4 wfrag_t(const float *W, int ld, int row, int k) {
    return pack4(*reinterpret_cast<const f32x4 *>(W + row * ld + k));
}
__device__ __forceinline__ bf16x4 ld4(const u16 *p) { return *reinterpret_cast<const bf16x4 *>(p); }
__device__ __forceinline__ f32x4 ldf4(const float *p) { return *reinterpret_cast<const f32x4 *>(p); }

// T(row, col) of an LDS tile as the fragment (m or n = col0 + l % 16, k = row0 +
// 4 (l / 16) + q): the transposing LDS read turns 4 rows x 16 columns per group of
// 16 lanes, each lane naming 4 columns of one row.
__device__ __forceinline__ bf16x4 ld4_t(const Lane &L, const u16 *t, int pitch, int row0, int col0) {
    const u16 *p = t + (row0 + 4 * L.g + (L.r >> 2)) * pitch + col0 + 4 * (L.r & 3);
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) bf16x4 *)p);
}

// Rows of MLP inputs in 16 B chunks of 8 bfloat16.
struct ZNode {  // [a (64), b (64)]
    const u16 *a, *b;
    __device__ __forceinline__ uint4 operator()(int row, int c) const {
        const u16 *p = c < kH / 8 ? a + (size_t)row * kH + 8 * c : b + (size_t)row * kH + 8 * c - kH;
        return *reinterpret_cast<const uint4 *>(p);
    }
};
struct ZInput {  // the network's FP32 input
    const float *x;
    __device__ __forceinline__ uint4 operator()(int row, int c) const {
        const float *p = x + (size_t)row * kDin + 8 * c;
        const bf16x4 v[2] = {pack4(ldf4(p)), pack4(ldf4(p + 4))};
        return __builtin_bit_cast(uint4, v);
    }
};
struct ZMsg {  // [h_dst, h_src, f] of edge `row`
    const int *src, *dst;
    const u16 *hb, *f;
    __device__ __forceinline__ uint4 operator()(int row, int c) const {
        const u16 *p;
        if (c < kH / 8) p = hb + (size_t)dst[row] * kH + 8 * c;
        else if (c < kH / 4) p = hb + (size_t)src[row] * kH + 8 * c - kH;
        else p = f + (size_t)row * kDedge + 8 * c - 2 * kH;
        return *reinterpret_cast<const uint4 *>(p);
    }
};

// Rows row0 .. row0 + n of an MLP input into an LDS tile, zero behind them.
template <int K, typename Z>
__device__ __forceinline__ void load_z(const Z &z, int row0, int n, u16 *t) {
    constexpr int kC = K / 8;
    for (int k = threadIdx.x; k < kTileRows * kC; k += kT) {
        const int r = k / kC, c = k - r * kC;
        uint4 v = {0, 0, 0, 0};
        if (r < n) v = z(row0 + r, c);
        *reinterpret_cast<uint4 *>(t + r * (K + kPad) + 8 * c) = v;
    }
}

// Hidden layer of row block i of a tile: W1^T z + b1 for the wavefront's 16 units.
template <int K>
__device__ __forceinline__ f32x4 hidden(const Lane &L, const u16 *z, int i, const bf16x4 *w1, f32x4 b1) {
    f32x4 a = {0.f, 0.f, 0.f, 0.f};
    const u16 *row = z + (16 * i + L.r) * (K + kPad) + 4 * L.g;
#pragma unroll
    for (int k = 0; k < K / 16; k++) a = mfma(w1[k], ld4(row + 16 * k), a);
    return a + b1;
}

__device__ __forceinline__ f32x4 silu4(f32x4 a) { return f32x4{silu(a[0]), silu(a[1]), silu(a[2]), silu(a[3])}; }

// One layer: messages of the tile's edges, their mean per node, the update MLP and
// the residual sum.  Thread (node slot t / 16, columns 4 (t % 16) ..) sums its node's
// messages in edge order, over the chunks of kTileRows edges that a single node of
// higher degree takes.  agg (training): the mean, rounded as the update uses it.
// Bound by latency: a tile is a chain of dependent loads (node range, edge ends,
// states) and short products.  A layer of the 221,184-cell hex mesh (1.3M edges)
// takes 0.227 ms (0.252 with expf, the IEEE division and integer rounding; four
// wavefronts a SIMD, which the compiler would give up for instruction order); gathering, two products, mean and update as kernels of their own
// took 2.1 ms, most of it on the edge rows' way through memory.
__global__ __launch_bounds__(kT, 4) void k_layer_fwd(int tiles, const int *__restrict__ tile_n0,
                                                  const int *__restrict__ in_off, ZMsg zm,
                                                  const float *__restrict__ inv_deg, const float *__restrict__ h,
                                                  float *__restrict__ h_out, u16 *__restrict__ hb_out,
                                                  u16 *__restrict__ agg, const float *__restrict__ wm,
                                                  const float *__restrict__ wu) {
    constexpr int kZ = kKmsg + kPad, kS = kH + kPad, kU = kKupd + kPad, kM = kH + 4;
    static_assert(kM * 4 <= kZ * 2, "the messages take the place of the edge rows");
    __shared__ __align__(16) u16 z[kTileRows * kZ], s1[kTileRows * kS], u[kTileNodes * kU], t1[kTileNodes * kS];
    float *msg = reinterpret_cast<float *>(z);
    const Lane L;
    const int j = 16 * L.w + L.r, j0 = 16 * L.w + 4 * L.g;
    const float *m2 = wm + kKmsg * kH + kH, *v2 = wu + kKupd * kH + kH;
    bf16x4 w1[kKmsg / 16], w2[kH / 16], u1[kKupd / 16], u2[kH / 16];
#pragma unroll
    for (int k = 0; k < kKmsg / 16; k++) w1[k] = wfrag(wm, kH, j, 16 * k + 4 * L.g);
#pragma unroll
    for (int k = 0; k < kKupd / 16; k++) u1[k] = wfrag(wu, kH, j, 16 * k + 4 * L.g);
#pragma unroll
    for (int k = 0; k < kH / 16; k++) {
        w2[k] = wfrag(m2, kH, j, 16 * k + 4 * L.g);
        u2[k] = wfrag(v2, kH, j, 16 * k + 4 * L.g);
    }
    const f32x4 mb1 = ldf4(m2 - kH + j0), mb2 = ldf4(m2 + kH * kH + j0);
    const f32x4 ub1 = ldf4(v2 - kH + j0), ub2 = ldf4(v2 + kH * kH + j0);
    const int slot = threadIdx.x >> 4, col = 4 * (threadIdx.x & 15);
    for (int t = blockIdx.x; t < tiles; t += gridDim.x) {
        const int n0 = tile_n0[t], nn = tile_n0[t + 1] - n0;
        const int e0 = in_off[n0], e1 = in_off[n0 + nn];
        const bool mine = slot < nn;
        const int p0 = mine ? in_off[n0 + slot] : e1, p1 = mine ? in_off[n0 + slot + 1] : e1;
        f32x4 sum = {0.f, 0.f, 0.f, 0.f};
        for (int eb = e0; eb < e1; eb += kTileRows) {
            const int ne = min(kTileRows, e1 - eb);
            load_z<kKmsg>(zm, eb, ne, z);
            __syncthreads();
#pragma unroll
            for (int i = 0; i < kTileRows / 16; i++)
                if (16 * i < ne)
                    *reinterpret_cast<bf16x4 *>(s1 + (16 * i + L.r) * kS + j0) =
                        pack4(silu4(hidden<kKmsg>(L, z, i, w1, mb1)));
            __syncthreads();
#pragma unroll
            for (int i = 0; i < kTileRows / 16; i++)
                if (16 * i < ne)
                    *reinterpret_cast<f32x4 *>(msg + (16 * i + L.r) * kM + j0) = hidden<kH>(L, s1, i, w2, mb2);
            __syncthreads();
            for (int e = max(p0, eb); e < min(p1, eb + ne); e++) sum += ldf4(msg + (e - eb) * kM + col);
            __syncthreads();
        }
        if (mine) {
            const int n = n0 + slot;
            const bf16x4 a = pack4(sum * inv_deg[n]);
            *reinterpret_cast<bf16x4 *>(u + slot * kU + kH + col) = a;
            *reinterpret_cast<bf16x4 *>(u + slot * kU + col) = ld4(zm.hb + (size_t)n * kH + col);
            if (agg) *reinterpret_cast<bf16x4 *>(agg + (size_t)n * kH + col) = a;
        }
        __syncthreads();
        *reinterpret_cast<bf16x4 *>(t1 + L.r * kS + j0) = pack4(silu4(hidden<kKupd>(L, u, 0, u1, ub1)));
        __syncthreads();
        const f32x4 d = hidden<kH>(L, t1, 0, u2, ub2);
        if (L.r < nn) {
            const size_t at = (size_t)(n0 + L.r) * kH + j0;
            const f32x4 hn = d + ldf4(h + at);
            *reinterpret_cast<f32x4 *>(h_out + at) = hn;
            *reinterpret_cast<bf16x4 *>(hb_out + at) = pack4(hn);
        }
    }
}

// out = W2 silu(W1 z + b1) + b2 of node rows (encoder, decoder); ob: a bfloat16 copy.
template <int K, int O, typename Z>
__global__ __launch_bounds__(kT) void k_node_fwd(int rows, Z zs, const float *__restrict__ w, float *__restrict__ out,
                                                 u16 *__restrict__ ob) {
    constexpr int kS = kH + kPad;
    __shared__ __align__(16) u16 z[kTileRows * (K + kPad)], s1[kTileRows * kS];
    const Lane L;
    const int j0 = 16 * L.w + 4 * L.g;
    const float *W2 = w + K * kH + kH;
    // 16 outputs: the wavefronts share the row blocks instead
    const int m0 = O == 16 ? 0 : 16 * L.w;
    bf16x4 w1[K / 16], w2[kH / 16];
#pragma unroll
    for (int k = 0; k < K / 16; k++) w1[k] = wfrag(w, kH, 16 * L.w + L.r, 16 * k + 4 * L.g);
#pragma unroll
    for (int k = 0; k < kH / 16; k++) w2[k] = wfrag(W2, O, m0 + L.r, 16 * k + 4 * L.g);
    const f32x4 b1 = ldf4(W2 - kH + j0), b2 = ldf4(W2 + kH * O + m0 + 4 * L.g);
    for (int row0 = blockIdx.x * kTileRows; row0 < rows; row0 += gridDim.x * kTileRows) {
        const int n = min(kTileRows, rows - row0);
        load_z<K>(zs, row0, n, z);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kTileRows / 16; i++)
            *reinterpret_cast<bf16x4 *>(s1 + (16 * i + L.r) * kS + j0) = pack4(silu4(hidden<K>(L, z, i, w1, b1)));
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kTileRows / 16; i++) {
            if (O == 16 && i != L.w) continue;
            const f32x4 v = hidden<kH>(L, s1, i, w2, b2);
            if (16 * i + L.r < n) {
                const size_t at = (size_t)(row0 + 16 * i + L.r) * O + m0 + 4 * L.g;
                *reinterpret_cast<f32x4 *>(out + at) = v;
                if (ob) *reinterpret_cast<bf16x4 *>(ob + at) = pack4(v);
            }
        }
    }
}

// Backward of one MLP over tiles of kTileRows rows: z (input) and dy (gradient of the
// output) in LDS, parameter gradients in registers until store().  NZ: 16-column
// blocks of the input gradient that are wanted.
template <int K, int O, int NZ>
struct MlpBwd {
    static constexpr int kZ = K + kPad, kS = kH + kPad, kY = O + kPad, kX = (NZ + 3) / 4;
    struct Lds {
        __align__(16) u16 z[kTileRows * kZ], dy[kTileRows * kY], s1[kTileRows * kS], da[kTileRows * kS];
    };
    Lane L;
    bf16x4 w1[K / 16], w2t[O / 16], w1t[kX > 0 ? kX : 1][kH / 16];
    f32x4 b1, dW1[K / 16], dW2[O / 16], db1, db2;

    __device__ __forceinline__ MlpBwd(const float *w) {
        const float *W2 = w + K * kH + kH;
        const int j = 16 * L.w + L.r;
#pragma unroll
        for (int k = 0; k < K / 16; k++) w1[k] = wfrag(w, kH, j, 16 * k + 4 * L.g);
#pragma unroll
        for (int k = 0; k < O / 16; k++) w2t[k] = wfrag_t(W2, O, j, 16 * k + 4 * L.g);
#pragma unroll
        for (int x = 0; x < kX; x++)
#pragma unroll
            for (int k = 0; k < kH / 16; k++)
                w1t[x][k] = wfrag_t(w, kH, 16 * (L.w + 4 * x) + L.r, 16 * k + 4 * L.g);
        b1 = ldf4(W2 - kH + 16 * L.w + 4 * L.g);
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < K / 16; k++) dW1[k] = zero;
#pragma unroll
        for (int k = 0; k < O / 16; k++) dW2[k] = zero;
        db1 = db2 = zero;
    }

    // The tile's output gradients, rounded, zero behind its n rows; a thread keeps to
    // four columns, whose unrounded sum is the gradient of b2.
    template <typename DY>
    __device__ __forceinline__ void load_dy(const DY &dy, int row0, int n, u16 *t) {
        constexpr int kC = O / 4;
        const int c = threadIdx.x % kC;
#pragma unroll
        for (int i = 0; i < kTileRows * kC / kT; i++) {
            const int r = threadIdx.x / kC + i * (kT / kC);
            f32x4 v = {0.f, 0.f, 0.f, 0.f};
            if (r < n) v = dy(row0 + r, 4 * c);
            db2 += v;
            *reinterpret_cast<bf16x4 *>(t + r * kY + 4 * c) = pack4(v);
        }
    }

    // After load_z, load_dy and a barrier: the hidden layer again, its gradient da,
    // and the tile's share of the parameter gradients.  Leaves da in LDS, z and dy
    // free behind the barrier at the end.
    __device__ __forceinline__ void tile(Lds &s) {
        const int j0 = 16 * L.w + 4 * L.g;
#pragma unroll 1  // (registers)
        for (int i = 0; i < kTileRows / 16; i++) {
            const f32x4 a = hidden<K>(L, s.z, i, w1, b1);
            const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
            const f32x4 ds = hidden<O>(L, s.dy, i, w2t, zero);
            const f32x4 d = {ds[0] * dsilu(a[0]), ds[1] * dsilu(a[1]), ds[2] * dsilu(a[2]), ds[3] * dsilu(a[3])};
            db1 += d;
            *reinterpret_cast<bf16x4 *>(s.s1 + (16 * i + L.r) * kS + j0) = pack4(silu4(a));
            *reinterpret_cast<bf16x4 *>(s.da + (16 * i + L.r) * kS + j0) = pack4(d);
        }
        __syncthreads();
#pragma unroll 1
        for (int k = 0; k < kTileRows / 16; k++) {
            const bf16x4 hs = ld4_t(L, s.s1, kS, 16 * k, 16 * L.w), hd = ld4_t(L, s.da, kS, 16 * k, 16 * L.w);
#pragma unroll
            for (int o = 0; o < O / 16; o++) dW2[o] = mfma(hs, ld4_t(L, s.dy, kY, 16 * k, 16 * o), dW2[o]);
#pragma unroll
            for (int c = 0; c < K / 16; c++) dW1[c] = mfma(ld4_t(L, s.z, kZ, 16 * k, 16 * c), hd, dW1[c]);
        }
        __syncthreads();
    }

    // Gradient of input columns 16 (wavefront + 4 x) + 4 (l / 16) .. of row 16 i + l % 16.
    __device__ __forceinline__ f32x4 dz(const Lds &s, int i, int x) const {
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        return hidden<kH>(L, s.da, i, w1t[x], zero);
    }

    // The block's partial gradients in the order of the parameters.
    __device__ __forceinline__ void store(Lds &s, float *part) {
        float *pb1 = part + K * kH, *pW2 = pb1 + kH, *pb2 = pW2 + kH * O;
#pragma unroll
        for (int c = 0; c < K / 16; c++)
#pragma unroll
            for (int q = 0; q < 4; q++) part[(16 * c + 4 * L.g + q) * kH + 16 * L.w + L.r] = dW1[c][q];
#pragma unroll
        for (int o = 0; o < O / 16; o++)
#pragma unroll
            for (int q = 0; q < 4; q++) pW2[(16 * L.w + 4 * L.g + q) * O + 16 * o + L.r] = dW2[o][q];
#pragma unroll
        for (int off = 8; off > 0; off >>= 1)
#pragma unroll
            for (int q = 0; q < 4; q++) db1[q] += __shfl_xor(db1[q], off, 64);
        if (L.r == 0)
#pragma unroll
            for (int q = 0; q < 4; q++) pb1[16 * L.w + 4 * L.g + q] = db1[q];
        constexpr int kC = O / 4;
        static_assert(sizeof(s.s1) >= kT * sizeof(f32x4), "the sums over b2 take s1's place");
        f32x4 *red = reinterpret_cast<f32x4 *>(s.s1);
        __syncthreads();
        red[threadIdx.x] = db2;
        __syncthreads();
        if ((int)threadIdx.x < kC) {
            f32x4 v = red[threadIdx.x];
            for (int t = threadIdx.x + kC; t < kT; t += kC) v += red[t];
            *reinterpret_cast<f32x4 *>(pb2 + 4 * threadIdx.x) = v;
        }
    }
};

struct DyNode {
    const float *dy;
    int ld;
    __device__ __forceinline__ f32x4 operator()(int row, int c) const { return ldf4(dy + (size_t)row * ld + c); }
};
struct DyMsg {  // the mean's gradient: du[dst, 64:128] / deg
    const int *dst;
    const float *du, *inv_deg;
    __device__ __forceinline__ f32x4 operator()(int row, int c) const {
        const int d = dst[row];
        return ldf4(du + (size_t)d * kKupd + kH + c) * inv_deg[d];
    }
};

// Backward of an MLP on node rows: its gradient partials and, with NZ, dz [rows, 16 NZ].
template <int K, int O, int NZ, typename Z>
__global__ __launch_bounds__(kT, 2) void k_node_bwd(int rows, Z zs, DyNode dy, const float *__restrict__ w,
                                                 float *__restrict__ dz, float *__restrict__ part, size_t part_ld) {
    using B = MlpBwd<K, O, NZ>;
    __shared__ typename B::Lds s;
    B m(w);
    for (int row0 = blockIdx.x * kTileRows; row0 < rows; row0 += gridDim.x * kTileRows) {
        const int n = min(kTileRows, rows - row0);
        load_z<K>(zs, row0, n, s.z);
        m.load_dy(dy, row0, n, s.dy);
        __syncthreads();
        m.tile(s);
#pragma unroll
        for (int x = 0; x < B::kX; x++)
#pragma unroll 1
            for (int i = 0; i < kTileRows / 16; i++) {
                const f32x4 v = m.dz(s, i, x);
                if (16 * i + m.L.r < n)
                    *reinterpret_cast<f32x4 *>(dz + (size_t)(row0 + 16 * i + m.L.r) * (16 * NZ) +
                                               16 * (m.L.w + 4 * x) + 4 * m.L.g) = v;
            }
    }
    m.store(s, part + blockIdx.x * part_ld);
}

// Backward of the message MLP over the tiles of k_layer_fwd: its gradient partials, the
// source half of the input gradient per edge (dzs, summed by k_dh_out), and
//   dh[t] += du[t, 0:64] + sum_{e in in(t)} dz[e, 0:64].
// 383k edges: 0.167 ms with two blocks a CU (what the registers allow), 0.284 with
// one.  The kernels that this one stands for took 4 ms, 3 of them in weight
// gradients whose few blocks each walked 4096 rows.
__global__ __launch_bounds__(kT, 2) void k_msg_bwd(int tiles, const int *__restrict__ tile_n0,
                                                const int *__restrict__ in_off, ZMsg zm, DyMsg dy,
                                                const float *__restrict__ w, float *__restrict__ dh,
                                                float *__restrict__ dzs, float *__restrict__ part, size_t part_ld) {
    using B = MlpBwd<kKmsg, kH, 2 * kH / 16>;
    constexpr int kM = kH + 4;
    static_assert(kM * 4 <= B::kZ * 2, "the destination half takes the place of the edge rows");
    __shared__ typename B::Lds s;
    float *dzd = reinterpret_cast<float *>(s.z);
    B m(w);
    const int slot = threadIdx.x >> 4, col = 4 * (threadIdx.x & 15);
    for (int t = blockIdx.x; t < tiles; t += gridDim.x) {
        const int n0 = tile_n0[t], nn = tile_n0[t + 1] - n0;
        const int e0 = in_off[n0], e1 = in_off[n0 + nn];
        const bool mine = slot < nn;
        const int p0 = mine ? in_off[n0 + slot] : e1, p1 = mine ? in_off[n0 + slot + 1] : e1;
        const size_t at = (size_t)(n0 + slot) * kH + col;
        f32x4 sum = {0.f, 0.f, 0.f, 0.f};
        if (mine) sum = ldf4(dh + at) + ldf4(dy.du + (size_t)(n0 + slot) * kKupd + col);
        for (int eb = e0; eb < e1; eb += kTileRows) {
            const int ne = min(kTileRows, e1 - eb);
            load_z<kKmsg>(zm, eb, ne, s.z);
            m.load_dy(dy, eb, ne, s.dy);
            __syncthreads();
            m.tile(s);
#pragma unroll 1
            for (int i = 0; i < kTileRows / 16; i++) {
                const int r = 16 * i + m.L.r, c = 16 * m.L.w + 4 * m.L.g;
                *reinterpret_cast<f32x4 *>(dzd + r * kM + c) = m.dz(s, i, 0);
                const f32x4 v = m.dz(s, i, 1);
                if (r < ne) *reinterpret_cast<f32x4 *>(dzs + (size_t)(eb + r) * kH + c) = v;
            }
            __syncthreads();
            for (int e = max(p0, eb); e < min(p1, eb + ne); e++) sum += ldf4(dzd + (e - eb) * kM + col);
            __syncthreads();
        }
        if (mine) *reinterpret_cast<f32x4 *>(dh + at) = sum;
    }
    m.store(s, part + blockIdx.x * part_ld);
}

//   dh[t] += sum_{e in out(t)} dzs[e]
__global__ __launch_bounds__(kT) void k_dh_out(int N, const int *__restrict__ out_off, const int *__restrict__ out_edge,
                                               const float *__restrict__ dzs, float *__restrict__ dh) {
    const int64_t t = (int64_t)blockIdx.x * kT + threadIdx.x;
    if (t >= (int64_t)N * (kH / 4)) return;
    const int i = (int)(t / (kH / 4)), c = 4 * (int)(t - (int64_t)i * (kH / 4));
    f32x4 s = ldf4(dh + (size_t)i * kH + c);
    for (int q = out_off[i]; q < out_off[i + 1]; q++) s += ldf4(dzs + (size_t)out_edge[q] * kH + c);
    *reinterpret_cast<f32x4 *>(dh + (size_t)i * kH + c) = s;
}

// g[p] = sum over the blocks' partials of parameter p, in a fixed order (four
// interleaved sums, then their sum).  Message MLPs have parts_e partials, the
// others parts_n.
constexpr int kEnc = (kDin + 1) * kH + (kH + 1) * kH;
constexpr int kMsg = (kKmsg + 1) * kH + (kH + 1) * kH;
constexpr int kUpd = (kKupd + 1) * kH + (kH + 1) * kH;

__global__ __launch_bounds__(kT) void k_sum_parts(int P, int parts_n, int parts_e, const float *__restrict__ part,
                                                  float *__restrict__ g) {
    __shared__ float red[4][64];
    const int o = threadIdx.x & 63, sl = threadIdx.x >> 6;
    const int p = blockIdx.x * 64 + o;
    float s = 0.f;
    if (p < P) {
        const int q = p - kEnc;
        const bool msg = q >= 0 && q < kLayers * (kMsg + kUpd) && q % (kMsg + kUpd) < kMsg;
        const int n = msg ? parts_e : parts_n;
#pragma unroll 8
        for (int b = sl; b < n; b += 4) s += part[(size_t)b * P + p];
    }
    red[sl][o] = s;
    __syncthreads();
    if (sl == 0 && p < P) g[p] = (red[0][o] + red[1][o]) + (red[2][o] + red[3][o]);
}

// dy = 2 (y - t) mask / n_used; per-block partial sums of the squared error
__global__ __launch_bounds__(kT) void k_mse(int64_t n, float inv_n, const float *__restrict__ y,
                                            const float *__restrict__ tgt, const float *__restrict__ mask,
                                            float *__restrict__ dy, double *__restrict__ part) {
    __shared__ double red[kT];
    const int64_t i = (int64_t)blockIdx.x * kT + threadIdx.x;
    double s = 0;
    if (i < n) {
        const float d = (y[i] - tgt[i]) * mask[i];
        dy[i] = 2.f * d * inv_n;
        s = (double)d * d;
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int off = kT / 2; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(kT) void k_adam(int n, float lr, float b1, float b2, float eps, float c1, float c2,
                                             const float *__restrict__ g, float *__restrict__ w,
                                             float *__restrict__ mo, float *__restrict__ ve) {
    const int i = blockIdx.x * kT + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float m = b1 * mo[i] + (1.f - b1) * gi;
    const float v = b2 * ve[i] + (1.f - b2) * gi * gi;
    mo[i] = m;
    ve[i] = v;
    w[i] -= lr * (m * c1) / (sqrtf(v * c2) + eps);
}

}  // namespace

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------

namespace {

struct MlpShape {
    int k, o;
};

MlpShape mlp_shape(int q) {
    if (q == 0) return {kDin, kH};
    if (q == kMlps - 1) return {kH, kDout};
    return (q % 2 == 1) ? MlpShape{kKmsg, kH} : MlpShape{kKupd, kH};
}

// offsets of W1, b1, W2, b2 of MLP q in the flat parameter vector
struct MlpOff {
    size_t W1, b1, W2, b2, end;
};

MlpOff mlp_off(int q) {
    size_t p = 0;
    for (int r = 0; r < q; r++) {
        const MlpShape s = mlp_shape(r);
        p += (size_t)s.k * kH + kH + (size_t)kH * s.o + s.o;
    }
    const MlpShape s = mlp_shape(q);
    MlpOff o;
    o.W1 = p;
    o.b1 = o.W1 + (size_t)s.k * kH;
    o.W2 = o.b1 + kH;
    o.b2 = o.W2 + (size_t)kH * s.o;
    o.end = o.b2 + s.o;
    return o;
}

size_t n_params_total() { return mlp_off(kMlps - 1).end; }

}  // namespace

struct plbfs_mpnn {
    int N = 0, E = 0;
    hipStream_t stream = nullptr;
    std::vector<void *> allocs;
    int *src = nullptr, *dst = nullptr, *in_off = nullptr, *out_off = nullptr, *out_edge = nullptr;
    float *inv_deg = nullptr;
    std::vector<int32_t> h_order;  // sorted edge -> caller edge
    size_t P = 0;
    float *w = nullptr, *g = nullptr, *m1 = nullptr, *m2 = nullptr;
    int adam_t = 0;
    int tiles = 0;            // edge tiles: nodes tile_n0[t] .. tile_n0[t + 1]
    int *tile_n0 = nullptr;
    float *x = nullptr, *y = nullptr, *tgt = nullptr, *mask = nullptr, *dy = nullptr;
    float *h[2] = {};                // node states, ping-pong over the layers
    u16 *hb[kLayers + 1] = {};       // ... as bfloat16, of every layer (two in turn without training)
    u16 *agg[kLayers] = {};          // training: mean messages as bfloat16
    u16 *fb = nullptr;               // edge inputs as bfloat16
    float *dh = nullptr, *du = nullptr, *dzs = nullptr;  // backward scratch
    float *part = nullptr;           // [max(parts_n, parts_e)][P] weight-gradient partials
    int parts_n = 0, parts_e = 0;
    double *mse_part = nullptr;
    int mse_blocks = 0;
    float mse_scale = 1.f;
    bool train = false;
};

namespace {

int malloc_t(plbfs_mpnn *n, void **p, size_t bytes) {
    if (bytes == 0) bytes = 8;
    HIP_TRY(hipMalloc(p, bytes));
    n->allocs.push_back(*p);
    return PLBFS_OK;
}

template <typename T>
int upload_t(plbfs_mpnn *n, T **dst, const std::vector<T> &src) {
    int rc = malloc_t(n, (void **)dst, src.size() * sizeof(T));
    if (rc) return rc;
    if (!src.empty()) HIP_TRY(hipMemcpy(*dst, src.data(), src.size() * sizeof(T), hipMemcpyHostToDevice));
    return PLBFS_OK;
}

inline dim3 grid1(int64_t n) { return dim3((unsigned)((n + kT - 1) / kT)); }

// Blocks of a kernel over `tiles` tiles: enough to fill the chip a few times, each
// keeping its weights for several tiles where there are more.
inline dim3 tile_grid(int tiles, int most) { return dim3((unsigned)std::max(1, std::min(tiles, most))); }
inline int row_tiles(int rows) { return (rows + kTileRows - 1) / kTileRows; }
constexpr int kFwdBlocks = 1024;

ZMsg zmsg(const plbfs_mpnn *n, int layer) { return ZMsg{n->src, n->dst, n->hb[layer], n->fb}; }

void forward(plbfs_mpnn *n) {
    const int N = n->N, nt = row_tiles(N);
    hipLaunchKernelGGL((k_node_fwd<kDin, kH, ZInput>), tile_grid(nt, kFwdBlocks), dim3(kT), 0, n->stream, N,
                       ZInput{n->x}, n->w + mlp_off(0).W1, n->h[0], n->hb[0]);
    for (int l = 0; l < kLayers; l++)
        hipLaunchKernelGGL(k_layer_fwd, tile_grid(n->tiles, kFwdBlocks), dim3(kT), 0, n->stream, n->tiles, n->tile_n0,
                           n->in_off, zmsg(n, l), n->inv_deg, n->h[l & 1], n->h[(l + 1) & 1], n->hb[l + 1],
                           n->agg[l], n->w + mlp_off(1 + 2 * l).W1, n->w + mlp_off(2 + 2 * l).W1);
    hipLaunchKernelGGL((k_node_fwd<kH, kDout, ZNode>), tile_grid(nt, kFwdBlocks), dim3(kT), 0, n->stream, N,
                       ZNode{n->hb[kLayers], nullptr}, n->w + mlp_off(kMlps - 1).W1, n->y, (u16 *)nullptr);
}

void backward(plbfs_mpnn *n) {
    const int N = n->N;
    const size_t P = n->P;
    const dim3 gn(n->parts_n), ge(n->parts_e), block(kT);
    hipStream_t st = n->stream;
    auto part = [&](int q) { return n->part + mlp_off(q).W1; };
    auto w = [&](int q) { return n->w + mlp_off(q).W1; };
    hipLaunchKernelGGL((k_node_bwd<kH, kDout, kH / 16, ZNode>), gn, block, 0, st, N, ZNode{n->hb[kLayers], nullptr},
                       DyNode{n->dy, kDout}, w(kMlps - 1), n->dh, part(kMlps - 1), P);
    for (int l = kLayers - 1; l >= 0; l--) {
        const int qm = 1 + 2 * l, qu = 2 + 2 * l;
        hipLaunchKernelGGL((k_node_bwd<kKupd, kH, kKupd / 16, ZNode>), gn, block, 0, st, N,
                           ZNode{n->hb[l], n->agg[l]}, DyNode{n->dh, kH}, w(qu), n->du, part(qu), P);
        hipLaunchKernelGGL(k_msg_bwd, ge, block, 0, st, n->tiles, n->tile_n0, n->in_off, zmsg(n, l),
                           DyMsg{n->dst, n->du, n->inv_deg}, w(qm), n->dh, n->dzs, part(qm), P);
        hipLaunchKernelGGL(k_dh_out, grid1((int64_t)N * (kH / 4)), block, 0, st, N, n->out_off, n->out_edge, n->dzs,
                           n->dh);
    }
    hipLaunchKernelGGL((k_node_bwd<kDin, kH, 0, ZInput>), gn, block, 0, st, N, ZInput{n->x}, DyNode{n->dh, kH}, w(0),
                       (float *)nullptr, part(0), P);
    hipLaunchKernelGGL(k_sum_parts, dim3((unsigned)((P + 63) / 64)), block, 0, st, (int)P, n->parts_n, n->parts_e,
                       n->part, n->g);
}

}  // namespace

extern "C" int plbfs_mpnn_n_params(void) { return (int)n_params_total(); }

extern "C" int plbfs_mpnn_create(int32_t n_nodes, int32_t n_edges, const int32_t *src, const int32_t *dst,
                                 const float *edge_feat, int32_t train, plbfs_mpnn **out) {
    if (!out || n_nodes <= 0 || n_edges < 0 || (n_edges > 0 && (!src || !dst || !edge_feat)))
        return plbfs_fail(PLBFS_ERR_INPUT, "bad graph");
    *out = nullptr;
    for (int e = 0; e < n_edges; e++)
        if (src[e] < 0 || src[e] >= n_nodes || dst[e] < 0 || dst[e] >= n_nodes)
            return plbfs_fail(PLBFS_ERR_INPUT, "edge %d: node index out of range", e);
    if (plbfs_device_count() <= 0) return plbfs_fail(PLBFS_ERR_NODEVICE, "no HIP device visible");
    auto *n = new plbfs_mpnn();
    auto fail = [&](int rc) {
        plbfs_mpnn_destroy(n);
        return rc;
    };
    const int N = n_nodes, E = n_edges;
    n->N = N;
    n->E = E;
    n->train = train != 0;
    if (hipStreamCreateWithFlags(&n->stream, hipStreamNonBlocking) != hipSuccess)
        return fail(plbfs_fail(PLBFS_ERR_HIP, "hipStreamCreate"));
    // sort edges by (dst, src), stable
    std::vector<int32_t> ord(E);
    std::iota(ord.begin(), ord.end(), 0);
    std::stable_sort(ord.begin(), ord.end(), [&](int a, int b) {
        return dst[a] != dst[b] ? dst[a] < dst[b] : src[a] < src[b];
    });
    n->h_order = ord;
    std::vector<int32_t> s(E), d(E), in_off(N + 1, 0), out_off(N + 1, 0), out_edge(E);
    std::vector<u16> f((size_t)E * kDedge);
    std::vector<float> inv_deg(N);
    for (int e = 0; e < E; e++) {
        s[e] = src[ord[e]];
        d[e] = dst[ord[e]];
        for (int k = 0; k < kDedge; k++) f[(size_t)e * kDedge + k] = to_bf16(edge_feat[(size_t)ord[e] * kDedge + k]);
        in_off[d[e] + 1]++;
        out_off[s[e] + 1]++;
    }
    for (int i = 0; i < N; i++) {
        inv_deg[i] = 1.0f / (float)std::max(in_off[i + 1], 1);
        in_off[i + 1] += in_off[i];
        out_off[i + 1] += out_off[i];
    }
    {
        std::vector<int32_t> fill(out_off.begin(), out_off.end() - 1);
        for (int e = 0; e < E; e++) out_edge[fill[s[e]]++] = e;  // increasing edge order per source
    }
    int rc;
    if ((rc = upload_t(n, &n->src, s)) || (rc = upload_t(n, &n->dst, d)) || (rc = upload_t(n, &n->in_off, in_off)) ||
        (rc = upload_t(n, &n->out_off, out_off)) || (rc = upload_t(n, &n->out_edge, out_edge)) ||
        (rc = upload_t(n, &n->inv_deg, inv_deg)) || (rc = upload_t(n, &n->fb, f)))
        return fail(rc);
    // edge tiles: nodes while they and their in-edges fit, at least one
    std::vector<int32_t> t0(1, 0);
    for (int i = 0; i < N;) {
        int k = i + 1;
        while (k < N && k - i < kTileNodes && in_off[k + 1] - in_off[i] <= kTileRows) k++;
        t0.push_back(k);
        i = k;
    }
    n->tiles = (int)t0.size() - 1;
    if ((rc = upload_t(n, &n->tile_n0, t0))) return fail(rc);
    n->P = n_params_total();
    const size_t P = n->P;
    std::vector<float> zero(P, 0.f);
    if ((rc = upload_t(n, &n->w, zero)) || (rc = upload_t(n, &n->g, zero)) || (rc = upload_t(n, &n->m1, zero)) ||
        (rc = upload_t(n, &n->m2, zero)))
        return fail(rc);
    auto fa = [&](float **p, size_t count) { return malloc_t(n, (void **)p, count * sizeof(float)); };
    auto ha = [&](u16 **p, size_t count) { return malloc_t(n, (void **)p, count * sizeof(u16)); };
    if ((rc = fa(&n->x, (size_t)N * kDin)) || (rc = fa(&n->y, (size_t)N * kDout)) ||
        (rc = fa(&n->tgt, (size_t)N * kDout)) || (rc = fa(&n->mask, (size_t)N * kDout)) ||
        (rc = fa(&n->dy, (size_t)N * kDout)) || (rc = fa(&n->h[0], (size_t)N * kH)) ||
        (rc = fa(&n->h[1], (size_t)N * kH)))
        return fail(rc);
    for (int l = 0; l <= kLayers; l++) {
        if (!n->train && l >= 2) {
            n->hb[l] = n->hb[l & 1];
            continue;
        }
        if ((rc = ha(&n->hb[l], (size_t)N * kH))) return fail(rc);
    }
    if (n->train) {
        n->parts_n = std::min(row_tiles(N), kMaxParts);
        n->parts_e = std::min(n->tiles, kMaxParts);
        for (int l = 0; l < kLayers; l++)
            if ((rc = ha(&n->agg[l], (size_t)N * kH))) return fail(rc);
        if ((rc = fa(&n->dh, (size_t)N * kH)) || (rc = fa(&n->du, (size_t)N * kKupd)) ||
            (rc = fa(&n->dzs, (size_t)E * kH)) || (rc = fa(&n->part, P * std::max(n->parts_n, n->parts_e))))
            return fail(rc);
    }
    n->mse_blocks = (int)(((int64_t)N * kDout + kT - 1) / kT);
    if ((rc = malloc_t(n, (void **)&n->mse_part, (size_t)n->mse_blocks * sizeof(double)))) return fail(rc);
    *out = n;
    return PLBFS_OK;
}

extern "C" int plbfs_mpnn_destroy(plbfs_mpnn *n) {
    if (!n) return PLBFS_OK;
    if (n->stream) hipStreamSynchronize(n->stream);
    for (void *p : n->allocs) hipFree(p);
    if (n->stream) hipStreamDestroy(n->stream);
    delete n;
    return PLBFS_OK;
}

extern "C" int plbfs_mpnn_set_params(plbfs_mpnn *n, const float *params) {
    if (!n || !params) return plbfs_fail(PLBFS_ERR_INPUT, "null argument");
    // on the network's stream, behind an Adam step that may still run
    HIP_TRY(hipMemcpyAsync(n->w, params, n->P * sizeof(float), hipMemcpyHostToDevice, n->stream));
    HIP_TRY(hipMemsetAsync(n->m1, 0, n->P * sizeof(float), n->stream));
    HIP_TRY(hipMemsetAsync(n->m2, 0, n->P * sizeof(float), n->stream));
    HIP_TRY(hipStreamSynchronize(n->stream));
    n->adam_t = 0;
    return PLBFS_OK;
}

extern "C" int plbfs_mpnn_get_params(plbfs_mpnn *n, float *params) {
    if (!n || !params) return plbfs_fail(PLBFS_ERR_INPUT, "null argument");
    HIP_TRY(hipStreamSynchronize(n->stream));
    HIP_TRY(hipMemcpy(params, n->w, n->P * sizeof(float), hipMemcpyDeviceToHost));
    return PLBFS_OK;
}

extern "C" int plbfs_mpnn_forward(plbfs_mpnn *n, const float *x, float *y) {
    if (!n || !x || !y) return plbfs_fail(PLBFS_ERR_INPUT, "null argument");
    HIP_TRY(hipMemcpyAsync(n->x, x, (size_t)n->N * kDin * sizeof(float), hipMemcpyHostToDevice, n->stream));
    forward(n);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpyAsync(y, n->y, (size_t)n->N * kDout * sizeof(float), hipMemcpyDeviceToHost, n->stream));
    HIP_TRY(hipStreamSynchronize(n->stream));
    return PLBFS_OK;
}

namespace {

int loss_grad_device(plbfs_mpnn *n, double *loss) {
    const int64_t ny = (int64_t)n->N * kDout;
    forward(n);
    hipLaunchKernelGGL(k_mse, grid1(ny), dim3(kT), 0, n->stream, ny, n->mse_scale, n->y, n->tgt, n->mask, n->dy,
                       n->mse_part);
    backward(n);
    HIP_TRY(hipGetLastError());
    if (loss) {
        std::vector<double> part(n->mse_blocks);
        HIP_TRY(hipMemcpyAsync(part.data(), n->mse_part, part.size() * sizeof(double), hipMemcpyDeviceToHost,
                               n->stream));
        HIP_TRY(hipStreamSynchronize(n->stream));
        double s = 0;
        for (double v : part) s += v;
        *loss = s * n->mse_scale;
    }
    return PLBFS_OK;
}

}  // namespace

extern "C" int plbfs_mpnn_loss_grad(plbfs_mpnn *n, const float *x, const float *target, const float *mask,
                                    double *loss, float *grads) {
    if (!n || !x || !target || !mask) return plbfs_fail(PLBFS_ERR_INPUT, "null argument");
    if (!n->train) return plbfs_fail(PLBFS_ERR_INPUT, "network created without training buffers");
    const size_t ny = (size_t)n->N * kDout;
    double used = 0;
    for (size_t i = 0; i < ny; i++) used += mask[i] != 0.f ? 1.0 : 0.0;
    n->mse_scale = (float)(1.0 / std::max(used, 1.0));
    HIP_TRY(hipMemcpyAsync(n->x, x, (size_t)n->N * kDin * sizeof(float), hipMemcpyHostToDevice, n->stream));
    HIP_TRY(hipMemcpyAsync(n->tgt, target, ny * sizeof(float), hipMemcpyHostToDevice, n->stream));
    HIP_TRY(hipMemcpyAsync(n->mask, mask, ny * sizeof(float), hipMemcpyHostToDevice, n->stream));
    int rc = loss_grad_device(n, loss);
    if (rc) return rc;
    // on the network's stream: without a loss to wait for, the kernels may still run
    if (grads)
        HIP_TRY(hipMemcpyAsync(grads, n->g, n->P * sizeof(float), hipMemcpyDeviceToHost, n->stream));
    HIP_TRY(hipStreamSynchronize(n->stream));
    return PLBFS_OK;
}

extern "C" int plbfs_mpnn_adam_step(plbfs_mpnn *n, float lr, float beta1, float beta2, float eps) {
    if (!n) return plbfs_fail(PLBFS_ERR_INPUT, "null argument");
    n->adam_t++;
    const float c1 = 1.f / (1.f - std::pow(beta1, (float)n->adam_t));
    const float c2 = 1.f / (1.f - std::pow(beta2, (float)n->adam_t));
    hipLaunchKernelGGL(k_adam, grid1((int64_t)n->P), dim3(kT), 0, n->stream, (int)n->P, lr, beta1, beta2, eps, c1, c2,
                       n->g, n->w, n->m1, n->m2);
    HIP_TRY(hipGetLastError());
    return PLBFS_OK;
}

extern "C" int plbfs_mpnn_train(plbfs_mpnn *n, int32_t n_samples, const float *X, const float *T, const float *mask,
                                int32_t epochs, float lr, uint64_t seed, double *loss_hist) {
    if (!n || n_samples <= 0 || !X || !T || !mask || epochs <= 0) return plbfs_fail(PLBFS_ERR_INPUT, "bad arguments");
    if (!n->train) return plbfs_fail(PLBFS_ERR_INPUT, "network created without training buffers");
    const size_t nx = (size_t)n->N * kDin, ny = (size_t)n->N * kDout;
    float *dX = nullptr, *dT = nullptr;
    int rc;
    if ((rc = malloc_t(n, (void **)&dX, nx * n_samples * sizeof(float))) ||
        (rc = malloc_t(n, (void **)&dT, ny * n_samples * sizeof(float))))
        return rc;
    HIP_TRY(hipMemcpy(dX, X, nx * n_samples * sizeof(float), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dT, T, ny * n_samples * sizeof(float), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(n->mask, mask, ny * sizeof(float), hipMemcpyHostToDevice));
    double used = 0;
    for (size_t i = 0; i < ny; i++) used += mask[i] != 0.f ? 1.0 : 0.0;
    n->mse_scale = (float)(1.0 / std::max(used, 1.0));
    std::vector<int> order(n_samples);
    std::iota(order.begin(), order.end(), 0);
    uint64_t st = seed ? seed : 0x9E3779B97F4A7C15ull;
    auto rnd = [&]() {
        st ^= st << 13;
        st ^= st >> 7;
        st ^= st << 17;
        return st;
    };
    auto release = [&]() {
        for (float *p : {dX, dT}) {
            n->allocs.erase(std::find(n->allocs.begin(), n->allocs.end(), (void *)p));
            hipFree(p);
        }
    };
    for (int ep = 0; ep < epochs; ep++) {
        for (int i = n_samples - 1; i > 0; i--) std::swap(order[i], order[rnd() % (uint64_t)(i + 1)]);
        const double lr_min = lr / 20.0, ph = epochs > 1 ? (double)ep / (epochs - 1) : 0.0;
        const float lr_ep = (float)(lr_min + 0.5 * (lr - lr_min) * (1.0 + std::cos(M_PI * ph)));
        double sum = 0;
        for (int k = 0; k < n_samples; k++) {
            const int sidx = order[k];
            HIP_TRY(hipMemcpyAsync(n->x, dX + nx * sidx, nx * sizeof(float), hipMemcpyDeviceToDevice, n->stream));
            HIP_TRY(hipMemcpyAsync(n->tgt, dT + ny * sidx, ny * sizeof(float), hipMemcpyDeviceToDevice, n->stream));
            double l = 0;
            if ((rc = loss_grad_device(n, &l)) || (rc = plbfs_mpnn_adam_step(n, lr_ep, 0.9f, 0.999f, 1e-8f))) {
                hipStreamSynchronize(n->stream);
                release();
                return rc;
            }
            sum += l;
        }
        if (loss_hist) loss_hist[ep] = sum / n_samples;
    }
    HIP_TRY(hipStreamSynchronize(n->stream));
    release();
    return PLBFS_OK;
}
