// Immersed-boundary kernels shared by the single-case solver (ibm.hip) and
// the batched solver (batch.hip).
//
// Per step, before the RK stages (src/Solver_gpu.cu:687-718):
//   k_ibm_nodes   one or four wavefronts per node: interpolate the node velocity
//                 from the step-start state (src/immersed_boundary_method.cu:13-90),
//                 move X = X0 + U dt (:244-295), spring force F = -k dA (X - X_ref)
//                 (:161-190), and the spreading normaliser at the new position;
//   k_ibm_spread  16 lanes per affected (cell, case) record: sum of the
//                 node forces over its pairs (:299-375).
// Weights are normalised per node, W_cn = delta V_c / sum delta V, which is the
// reference's formula on its uniform unit grid.  No atomics.
//
// For a batch, node k belongs to case node_case[k] and reads the state record
// cell * B + case; affected records carry their case in cp_case.  Nodes and
// records of a case whose case_done flag is set are skipped.
#pragma once
#include "lbfs_device.hpp"
#include "plbfs_hip.h"

namespace plbfs {
namespace {

constexpr int kIbmThreads = 256;
constexpr int kIbmUnroll = 4;  // pairs per lane whose loads are issued together
// Wavefronts per node: four where a node has this many candidate pairs or more by
// the mean cell volume, i.e. on meshes of cells smaller than the kernel width, one
// elsewhere.  (The choice follows from the mesh, not the number of nodes, so that a
// batch sums in the order of its cases' single runs.)  4.1M tets, 2,000 nodes of some
// 1,300 pairs, nodes and spreading together 54 -> 43 us a step; 83k tets, 400 nodes, 45 -> 21 us.
constexpr double kIbmWidePairs = 512.0;
constexpr int kIbmWide = kIbmThreads / 64;

// Side of the cube a node's candidate cells lie in, over the kernel width: support
// plus drift margin (one width) on both sides.
inline bool ibm_wide(int kernel, double h, int64_t n_cells, double volume) {
    const double side = 2.0 * h * ((kernel == PLBFS_DELTA_HAT2 ? 1.0 : 2.0) + 1.0);
    return side * side * side * (double)n_cells >= kIbmWidePairs * volume;
}

__device__ __forceinline__ double ibm_phi(int kernel, double r) {
    r = fabs(r);
    if (kernel == PLBFS_DELTA_HAT2) return r < 1.0 ? 1.0 - r : 0.0;
    // Peskin, "The immersed boundary method", Acta Numerica 11 (2002), 4-point function
    if (r <= 1.0) return (3.0 - 2.0 * r + sqrt(1.0 + 4.0 * r - 4.0 * r * r)) / 8.0;
    if (r <= 2.0) return (5.0 - 2.0 * r - sqrt(-7.0 + 12.0 * r - 4.0 * r * r)) / 8.0;
    return 0.0;
}

__device__ __forceinline__ double ibm_delta(int kernel, double ih, const double4 &c, const double X[3]) {
    return ibm_phi(kernel, (c.x - X[0]) * ih) * ibm_phi(kernel, (c.y - X[1]) * ih) *
           ibm_phi(kernel, (c.z - X[2]) * ih) * (ih * ih * ih);
}

__device__ __forceinline__ double wave_allsum(double x) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
    return x;
}

struct IbmArgs {
    int n, N, kernel;
    int B;  // cases per cell record (1 for a single case)
    double ih, dt, k_dA, margin;
    double *x, *x0, *xref, *vel, *force;
    double4 *fn;             // per node force and spreading normaliser, for the spreading
    const double *xc;        // [3][n] positions the candidate lists were built around
    int rebuild;             // 1: ask the host for new lists at half the margin (single case)
    const double *node_kdA;  // per-node k dA, or null for the scalar k_dA
    const int32_t *node_case;  // per-node case, or null (case 0)
    const int32_t *np_off, *np_cell;
    const int32_t *cp_cell, *cp_off;
    const int2 *cp_pair;     // (node, node-major pair index) of every cell-major entry
    const int32_t *cp_case;  // per affected record case, or null (case 0)
    double *pw;              // [n_pairs] kernel weight delta(x_c - X_k) at the current node position
    const int32_t *case_done;  // per-case freeze flags, or null
    int *case_status;          // per-case status, or null
    int n_affected;
    const double4 *geo;      // per cell centroid and volume
};

// Sums of a node's lanes in a fixed order: butterflies, then the wavefronts in turn.
template <int W, int M>
__device__ __forceinline__ void node_sums(double (&v)[M]) {
#pragma unroll
    for (int q = 0; q < M; q++) v[q] = wave_allsum(v[q]);
    if constexpr (W > 1) {
        __shared__ double red[W][M];
        if ((threadIdx.x & 63) == 0)
#pragma unroll
            for (int q = 0; q < M; q++) red[threadIdx.x >> 6][q] = v[q];
        __syncthreads();
#pragma unroll
        for (int q = 0; q < M; q++) {
            v[q] = red[0][q];
#pragma unroll
            for (int w = 1; w < W; w++) v[q] += red[w][q];
        }
    }
}

// Bound by latency: a chain of list, weights and cells, states, sums.  A lane takes
// kIbmUnroll of its pairs at a time and issues all their loads before the first use;
// cells are read once for both passes unless a node has more pairs than that.
template <typename SV, int W>
__global__ __launch_bounds__(kIbmThreads) void k_ibm_nodes(IbmArgs a, Ctrl *__restrict__ ctrl,
                                                           const SV *__restrict__ st) {
    constexpr int T = 64 * W;
    if constexpr (W > 1) {
        // one answer for the whole block: another block's node may stop the run
        __shared__ int stop;
        if (threadIdx.x == 0) stop = ctrl->done;
        __syncthreads();
        if (stop) return;
    } else {
        if (ctrl->done) return;
    }
    const int lane = threadIdx.x & (T - 1);
    const int k = blockIdx.x * (kIbmThreads / T) + (threadIdx.x / T);
    if (k >= a.n) return;
    const int b = a.node_case ? a.node_case[k] : 0;
    if (a.case_done && a.case_done[b]) return;
    const int n = a.n;
    const int p0 = a.np_off[k], p1 = a.np_off[k + 1];
    const bool once = p1 - p0 <= T * kIbmUnroll;
    double4 geo[kIbmUnroll];
    double s[4] = {0, 0, 0, 0};  // sum of w, w u, w v, w w
    // weights at the current position: computed at set-up or by the previous step's
    // second pass
    for (int pb = p0 + lane; pb < p1; pb += T * kIbmUnroll) {
        int c[kIbmUnroll];
        double d[kIbmUnroll];
        SV sc[kIbmUnroll];
#pragma unroll
        for (int u = 0; u < kIbmUnroll; u++) {
            const int p = pb + T * u;
            c[u] = p < p1 ? a.np_cell[p] : -1;
            d[u] = p < p1 ? a.pw[p] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < kIbmUnroll; u++) {
            if (c[u] >= 0) geo[u] = a.geo[c[u]];
            if (d[u] != 0.0) sc[u] = st[(size_t)c[u] * a.B + b];
        }
#pragma unroll
        for (int u = 0; u < kIbmUnroll; u++) {
            if (d[u] != 0.0) {
                const double wv = d[u] * geo[u].w;
                s[0] += wv;
                s[1] += wv * sc[u].y;
                s[2] += wv * sc[u].z;
                s[3] += wv * sc[u].w;
            }
        }
    }
    node_sums<W>(s);
    const double S = s[0];
    // a node with no cell in its support (S = 0) is an error below; it stays
    // where it is, so that only finite positions and forces are written
    const bool supported = S > 0.0;
    const double U[3] = {supported ? s[1] / S : 0.0, supported ? s[2] / S : 0.0, supported ? s[3] / S : 0.0};
    const double kdA = a.node_kdA ? a.node_kdA[k] : a.k_dA;
    double Xn[3], F[3], drift = 0;
#pragma unroll
    for (int q = 0; q < 3; q++) {
        const double x0 = a.x0[(size_t)q * n + k], xr = a.xref[(size_t)q * n + k];
        Xn[q] = x0 + U[q] * a.dt;
        F[q] = (-kdA * (Xn[q] - xr));
        drift = fmax(drift, fabs(Xn[q] - a.xc[(size_t)q * n + k]));
    }
    double s2[1] = {0};
    for (int pb = p0 + lane; pb < p1; pb += T * kIbmUnroll) {
#pragma unroll
        for (int u = 0; u < kIbmUnroll; u++)
            if (!once && pb + T * u < p1) geo[u] = a.geo[a.np_cell[pb + T * u]];
#pragma unroll
        for (int u = 0; u < kIbmUnroll; u++) {
            const int p = pb + T * u;
            if (p < p1) {
                const double d = ibm_delta(a.kernel, a.ih, geo[u], Xn);
                a.pw[p] = d;
                if (d != 0.0) s2[0] += d * geo[u].w;
            }
        }
    }
    node_sums<W>(s2);
    const double S2 = s2[0];
    if (lane == 0) {
#pragma unroll
        for (int q = 0; q < 3; q++) {
            a.x[(size_t)q * n + k] = Xn[q];
            a.x0[(size_t)q * n + k] = Xn[q];
            a.vel[(size_t)q * n + k] = U[q];
            a.force[(size_t)q * n + k] = F[q];
        }
        a.fn[k] = double4{F[0], F[1], F[2], S2};
        // past half the margin the lists are rebuilt around the new positions
        // after this step; past the margin they may miss cells: an error
        if (a.rebuild && drift > 0.5 * a.margin) ctrl->rebuild = 1;
        if (!supported || !(S2 > 0.0) || drift > a.margin) {
            if (a.case_status) {
                // batch: only this case stops
                a.case_status[b] = PLBFS_ERR_IBM;
            } else {
                ctrl->status = PLBFS_ERR_IBM;
                ctrl->done = 1;
            }
        }
    }
}

template <typename SV>
inline void launch_ibm_nodes(const IbmArgs &a, bool wide, hipStream_t stream, Ctrl *ctrl, const SV *st) {
    const int per = wide ? 1 : kIbmWide;  // nodes a block
    hipLaunchKernelGGL((wide ? k_ibm_nodes<SV, kIbmWide> : k_ibm_nodes<SV, 1>), dim3((a.n + per - 1) / per),
                       dim3(kIbmThreads), 0, stream, a, ctrl, st);
}

// Kernel weights of every pair at the nodes' current positions (set-up).
__global__ __launch_bounds__(kIbmThreads) void k_ibm_weights(IbmArgs a) {
    const int lane = threadIdx.x & 63;
    const int k = blockIdx.x * (kIbmThreads / 64) + (threadIdx.x >> 6);
    if (k >= a.n) return;
    const int n = a.n;
    const double X[3] = {a.x[k], a.x[(size_t)n + k], a.x[2 * (size_t)n + k]};
    for (int p = a.np_off[k] + lane; p < a.np_off[k + 1]; p += 64)
        a.pw[p] = ibm_delta(a.kernel, a.ih, a.geo[a.np_cell[p]], X);
}

// kSpreadLanes lanes per affected record (kSpreadPerBlock records per
// workgroup): the lanes stride over the record's pairs in node order and a fixed
// butterfly inside the lane group sums them, so every record's force has one
// summation order wherever it is spread from.  A record has a few dozen pairs
// (a node's Peskin-4 support spans 4^3 cells, its candidate list with the drift
// margin 6^3), so a whole wavefront per record would leave most lanes idle.
// fbody is [3][B*N] component-major over records.
constexpr int kSpreadLanes = 16;
constexpr int kSpreadUnroll = 4;
constexpr int kSpreadPerBlock = kIbmThreads / kSpreadLanes;

__device__ __forceinline__ double group_allsum(double x) {
#pragma unroll
    for (int off = kSpreadLanes / 2; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
    return x;
}

__global__ __launch_bounds__(kIbmThreads) void k_ibm_spread(IbmArgs a, const Ctrl *__restrict__ ctrl,
                                                            double *__restrict__ fbody) {
    if (ctrl->done) return;
    const int lane = threadIdx.x & (kSpreadLanes - 1);
    const int j = blockIdx.x * kSpreadPerBlock + (int)(threadIdx.x / kSpreadLanes);
    // every lane of a group has the same j and case, so a group leaves as a
    // whole and the shuffles below never read a lane that has left
    if (j >= a.n_affected) return;
    const int c = a.cp_cell[j];
    const int b = a.cp_case ? a.cp_case[j] : 0;
    if (a.case_done && a.case_done[b]) return;
    double f0 = 0, f1 = 0, f2 = 0;
    const int q0 = a.cp_off[j], q1 = a.cp_off[j + 1];
    // kSpreadUnroll pairs per lane at a time, loads first (as in k_ibm_nodes); weights
    // and nodes together, though most weights of a list are zero: the nodes' records
    // are few and near
    for (int pb = q0 + lane; pb < q1; pb += kSpreadLanes * kSpreadUnroll) {
        int2 e[kSpreadUnroll];
        double d[kSpreadUnroll];
        double4 fn[kSpreadUnroll];
#pragma unroll
        for (int u = 0; u < kSpreadUnroll; u++)
            if (pb + kSpreadLanes * u < q1) e[u] = a.cp_pair[pb + kSpreadLanes * u];
#pragma unroll
        for (int u = 0; u < kSpreadUnroll; u++) {
            d[u] = 0.0;
            if (pb + kSpreadLanes * u < q1) {
                d[u] = a.pw[e[u].y];  // at the node's new position
                fn[u] = a.fn[e[u].x];
            }
        }
#pragma unroll
        for (int u = 0; u < kSpreadUnroll; u++) {
            if (d[u] != 0.0) {
                const double q = d[u] / fn[u].w;
                f0 += fn[u].x * q;
                f1 += fn[u].y * q;
                f2 += fn[u].z * q;
            }
        }
    }
    f0 = group_allsum(f0);
    f1 = group_allsum(f1);
    f2 = group_allsum(f2);
    if (lane == 0) {
        const size_t NR = (size_t)a.N * a.B, r = (size_t)c * a.B + b;
        fbody[r] = f0;
        fbody[NR + r] = f1;
        fbody[2 * NR + r] = f2;
    }
}

}  // namespace
}  // namespace plbfs
