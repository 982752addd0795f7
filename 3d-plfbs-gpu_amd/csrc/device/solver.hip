// PLBFS solver on one MI355X (gfx950): kernels, context and the C-ABI of
// include/plbfs_hip.h.
//
// Per RK stage two kernels run back to back on the context's stream, on meshes below
// 65,536 cells one (k_stage) that does the work of both:
//   k_grad         one thread per cell: least-squares gradients of rho,u,v,w
//                  from the folded stencil weights (src/gradients.cpp:319-389);
//                  ghost neighbours are evaluated from the owner and its patch.
//   k_flux_update  one block per 64 to 256 Hilbert-consecutive cells: every face of the
//                  block is evaluated once into an LDS slot (border faces by both
//                  blocks), then each cell gathers its faces' slots in the
//                  reference face order and applies the RK stage update
//                  (src/Solver.cpp:286-438).  The last stage also writes the new
//                  solution, the next local time step (src/Solver.cpp:1693-1776)
//                  and per-block residual partial sums.
// After the fourth stage k_finalize sums the partials in a fixed order
// (src/residuals.cpp:35-44,139-147) and sets the stop flag on convergence,
// NaN or rho blow-up; every kernel returns immediately once the flag is set.
// No float atomics are used anywhere, so runs are bitwise reproducible.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "ctx.hpp"
#include "stage.hpp"

using namespace plbfs;

namespace {

constexpr int kFinalizeThreads = 256;

// ---------------------------------------------------------------------------
// Kernels
// ---------------------------------------------------------------------------

// Fluxes of flux block blk's face items into their LDS slots, four arrays of
// max_items; the caller's barrier follows.  With staging the block's own records
// are first copied into LDS behind the slots.
template <typename S, bool kStaged>
__device__ __forceinline__ void block_fluxes(const DevMesh<S> &m, const DevParams &prm, const V4<S> *st,
                                             const V4<S> *grad, double *lds, int blk) {
    const int e0 = m.blk_item_off[blk], e1 = m.blk_item_off[blk + 1];
    const int nslot = m.max_items;
    S *sF = reinterpret_cast<S *>(lds);
    V4<S> *sRec = reinterpret_cast<V4<S> *>(reinterpret_cast<char *>(lds) + staged_offset<S>(m.max_items));
    SideLoader<S, Rec1, kStaged> ld{st, grad, Rec1{}, sRec, blk * m.block_cells, 0, 1, 0};
    if constexpr (kStaged) {
        ld.nc = min(m.N, ld.c0 + m.block_cells) - ld.c0;
        stage_records<S>(st, grad, 0, 0, 1, ld.c0, ld.nc, sRec);
        __syncthreads();
    }
    for (int e = e0 + threadIdx.x; e < e1; e += kBlock) {
        S F[4];
        item_flux<S>(m, prm, load_item<S>(m, e), ld, prm.visc3_invgam, INFINITY, F);
#pragma unroll
        for (int q = 0; q < 4; q++) sF[q * nslot + (e - e0)] = F[q];
    }
}

// Gather entries face by face (see DevMesh::g_ent); conv turns the layout's entry.
template <typename T, typename F>
static std::vector<T> entries_by_face(const Layout &L, int max_ent, T none, F conv) {
    const size_t N = (size_t)L.N;
    std::vector<T> v(N * max_ent, none);
    for (size_t i = 0; i < N; i++)
        for (int k = L.g_off[i]; k < L.g_off[i + 1]; k++) v[(size_t)(k - L.g_off[i]) * N + i] = conv(L.g_ent[k]);
    return v;
}

// Face items in groups of 64 (see DevMesh::it_p).
template <typename S>
static std::vector<float4> pack_items(const Layout &L) {
    const size_t E = (size_t)L.n_items, K = kItemChunks<S>;
    std::vector<float4> v((E + 63) / 64 * 64 * K);
    for (size_t e = 0; e < E; e++) {
        const double *g = &L.it_geo[kGeoPerItem * e];
        float4 *p = &v[(e >> 6) * 64 * K + (e & 63)];
        S f[12];
        const int third = L.it_nbr[e] < 0 ? 0 : 8;  // the normal, or the neighbour's offset
        for (int a = 0; a < 3; a++) {
            f[a] = (S)(g[a] * g[3]);
            f[3 + a] = (S)g[5 + a];
            f[6 + a] = (S)g[third + a];
        }
        if (std::is_same<S, float>::value) f[9] = (S)g[4];
        const int32_t on[2] = {L.it_own[e], L.it_nbr[e]};
        std::memcpy(reinterpret_cast<char *>(f) + 16 * K - sizeof on, on, sizeof on);
        for (size_t k = 0; k < K; k++) std::memcpy(p + 64 * k, reinterpret_cast<const char *>(f) + 16 * k, 16);
    }
    return v;
}

// Neighbours and stencil weights of k_stage's places from their cells' (at creation: on the
// host it took a tenth of a 32k-cell solver's creation).
template <typename S>
__global__ __launch_bounds__(kBlock) void k_places(DevMesh<S> m, int32_t *__restrict__ nbr, float4 *__restrict__ w) {
    constexpr int kPer = 16 / sizeof(S), kPieces = (3 * kMaxSlots + kPer - 1) / kPer;
    const int p = blockIdx.x * kBlock + threadIdx.x;
    if (p >= m.n_places) return;
    const int c = m.loc_cell[p], cnt = c >= 0 ? m.st_cnt[c] : 0;
    for (int s = 0; s < kMaxSlots; s++)
        nbr[(size_t)s * m.n_places + p] = s < cnt ? m.st_nbr[(size_t)s * m.N + c] : kNoNbr;
    for (int k = 0; k < kPieces; k++) {
        S v[kPer];
        for (int u = 0; u < kPer; u++) {
            const int q = k * kPer + u;
            v[u] = q < 3 * cnt ? m.st_w[(size_t)q * m.N + c] : (S)0;
        }
        __builtin_memcpy(&w[(size_t)k * m.n_places + p], v, 16);
    }
}

// Bound by HBM: a state read, the stencil (28 B a slot in FP64) and the record
// written are 241 B a tet, 0.98 GB in 0.181 ms on 4.1M tets in FP64 (5.4 TB/s; 6.0 by
// the counters' 1.08 GB, part of it from the last-level cache, where a large copy reaches
// 4.75-5.1); 0.239 ms with each lane storing its own record.
template <typename S>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(6))) void k_grad(DevMesh<S> m, const Ctrl *__restrict__ ctrl,
                                                 const V4<S> *__restrict__ st, V4<S> *__restrict__ grad) {
    if (ctrl->done) return;
    const int c0 = xcd_block(blockIdx.x, gridDim.x, 1) * kBlock;
    const int i = c0 + threadIdx.x;
    S g[12];
    V4<S> si;
    const int nc = min(m.N - c0, kBlock);
    const bool live = i < m.N;
    // the block's own states, then its records
    constexpr int kChunks = kGradRec<S> * sizeof(V4<S>) / 16;
    __shared__ float4 lds[kBlock * kChunks];
    if (m.grad_stage) {
        // the block's own states in LDS: most stencil neighbours are in the block
        V4<S> *sSt = reinterpret_cast<V4<S> *>(lds);
        if (live) sSt[threadIdx.x] = st[i];
        __syncthreads();
        if (live) {
            lsq_grad<S>(m, i, StagedStates<S>{st, sSt, c0, nc}, g);
            si = sSt[threadIdx.x];
        }
        __syncthreads();
    } else if (live) {
        lsq_grad<S>(m, i, GlobalStates<S, Rec1>{st, Rec1{}}, g);
        si = st[i];
    }
    // records assembled in LDS, then stored by the block as one contiguous run:
    // lane by lane at the records' stride a store takes the address unit two to
    // three times as long
    if (live) {
        V4<S> *o = reinterpret_cast<V4<S> *>(lds) + kGradRec<S> * threadIdx.x;
        if constexpr (kGradOff<S> == 1) o[0] = si;
        o[kGradOff<S>] = V4<S>{g[0], g[1], g[2], g[3]};
        o[kGradOff<S> + 1] = V4<S>{g[4], g[5], g[6], g[7]};
        o[kGradOff<S> + 2] = V4<S>{g[8], g[9], g[10], g[11]};
    }
    __syncthreads();
    float4 *out = reinterpret_cast<float4 *>(grad) + (size_t)kChunks * c0;
#pragma unroll
    for (int k = 0; k < kChunks; k++) {
        const int t = threadIdx.x + k * kBlock;
        if (t < kChunks * nc) out[t] = lds[t];
    }
}

// Faces between two flux blocks, one thread per face: flux into the border
// array that both blocks' cells read in their gather.
template <typename S>
__global__ __launch_bounds__(kBlock) void k_flux_border(DevMesh<S> m, DevParams prm, const Ctrl *__restrict__ ctrl,
                                                        const V4<S> *__restrict__ st_in,
                                                        const V4<S> *__restrict__ grad) {
    if (ctrl->done) return;
    const int t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= m.n_border) return;
    const SideLoader<S, Rec1, false> ld{st_in, grad, Rec1{}, nullptr, 0, 0, 1, 0};
    S F[4];
    item_flux<S>(m, prm, load_item<S>(m, m.border0 + t), ld, prm.visc3_invgam, INFINITY, F);
    const size_t nbd = (size_t)m.n_border;
#pragma unroll
    for (int q = 0; q < 4; q++) m.bflux[q * nbd + t] = F[q];
}

// What a cell's update reads from global memory.
template <typename S>
struct CellIn {
    CellFaces<S> faces;
    RkIn<S> rk;
    double force[3];
};

template <typename S, bool kAhead>
__device__ __forceinline__ void load_rk(const DevMesh<S> &m, StageArgs sa, bool force, int i, const double4 *t0,
                                        const Acc<S> *t1, const double *dtl, const double *fbody, CellIn<S> &in) {
    in.rk = load_rk<S, kAhead>(m, sa, i, (size_t)i, t0, t1, dtl);
    if (force)
        for (int q = 0; q < 3; q++) in.force[q] = fbody[(size_t)q * m.N + i];
}

// Residual and RK stage of cell i; returns its error code.
template <typename S, bool kAhead>
__device__ __forceinline__ int cell_update(const DevMesh<S> &m, const DevParams &prm, StageArgs sa, const S *sF,
                                           bool force, int i, const CellIn<S> &in, V4<S> *__restrict__ st_out,
                                           double4 *__restrict__ t0, Acc<S> *__restrict__ t1,
                                           double *__restrict__ dtl, double sq[4], double &dt_next) {
    double R[4];
    gather_residual<S, kAhead>(m, i, in.faces, sF, m.max_items, 1, 0, R);
    if (force) {
        R[1] += in.force[0];
        R[2] += in.force[1];
        R[3] += in.force[2];
    }
    return rk_update<S, kAhead>(m, prm, prm.visc, sa, i, (size_t)i, in.rk, R, st_out, t0, t1, dtl, sq, dt_next);
}

template <typename S>
__device__ __forceinline__ bool block_force(const DevMesh<S> &m, const DevParams &prm, int blk) {
    return prm.use_body_force && (!m.blk_force || m.blk_force[blk]);
}

// Block blk's residual sums (last stage).
__device__ __forceinline__ void block_sums(StageArgs sa, int blk, const double sq[4], int err,
                                           double *__restrict__ partials) {
    if (sa.stage == 3) {
        __shared__ double red[kBlock / 64][5];
        const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
        double e = (double)err;
        double r0 = wave_sum(sq[0]), r1 = wave_sum(sq[1]), r2 = wave_sum(sq[2]), r3 = wave_sum(sq[3]);
        // error code: max over the wave
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) e = fmax(e, __shfl_xor(e, off, 64));
        if (lane == 0) {
            red[wv][0] = r0; red[wv][1] = r1; red[wv][2] = r2; red[wv][3] = r3; red[wv][4] = e;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            double s[5] = {0, 0, 0, 0, 0};
            for (int q = 0; q < kBlock / 64; q++) {
                for (int c = 0; c < 4; c++) s[c] += red[q][c];
                s[4] = fmax(s[4], red[q][4]);
            }
            for (int c = 0; c < 5; c++) partials[(size_t)blk * 5 + c] = s[c];
        }
    }
}

// 6 waves per SIMD in FP32 and 4 in FP64, the most that hold without spills (77
// and 126 VGPRs).
template <typename S>
constexpr int kFluxMinWaves = std::is_same<S, float>::value ? 6 : 4;

template <typename S, bool kStaged>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(kFluxMinWaves<S>))) void k_flux_update(
    DevMesh<S> m, DevParams prm, StageArgs sa, const Ctrl *__restrict__ ctrl, const V4<S> *__restrict__ st_in,
    const V4<S> *__restrict__ grad, V4<S> *__restrict__ st_out, double4 *__restrict__ t0, Acc<S> *__restrict__ t1,
    double *__restrict__ dtl, const double *__restrict__ fbody, double *__restrict__ partials) {
    extern __shared__ double lds[];
    if (ctrl->done) return;
    const int blk = xcd_block(blockIdx.x, gridDim.x, m.xcd_remap);
    const S *sF = reinterpret_cast<const S *>(lds);
    block_fluxes<S, kStaged>(m, prm, st_in, grad, lds, blk);
    __syncthreads();
    const bool force = block_force(m, prm, blk);
    double sq[4] = {0, 0, 0, 0};
    int err = 0;
    const int c_end = min(m.N, (blk + 1) * m.block_cells);
    for (int i = blk * m.block_cells + threadIdx.x; i < c_end; i += kBlock) {
        constexpr bool kAhead = std::is_same<S, double>::value;
        CellIn<S> in;
        in.faces = load_faces<S>(m, i);
        load_rk<S, kAhead>(m, sa, force, i, t0, t1, dtl, fbody, in);
        double dt;
        const int e = cell_update<S, kAhead>(m, prm, sa, sF, force, i, in, st_out, t0, t1, dtl, sq, dt);
        if (e == 1) err = 1;
        else if (e == 2 && err == 0) err = 2;
    }
    block_sums(sa, blk, sq, err, partials);
}

// One RK stage of a mesh of up to 1024 64-cell flux blocks: k_grad and k_flux_update in
// one kernel, with the gradients of every cell that the block's items read computed
// here, into LDS, by each block that reads them (some 160 for 64 hexes).  Such a mesh
// is bound by latencies and not by work: a launch and a round through memory saved are
// worth the repeated sums.  What depends on the block's and the thread's number alone
// (places, neighbours, weights, the first item, the cell's update) is loaded at the
// start, so that it arrives while the control block does; patches are read from LDS.
// Step in FP64, two kernels / one / one with these loads at the start: 216 hexes 52.4 /
// 46.0 / 35.5 us, 32k 89 / 67 / 51.5, 64k tets 106 / 107 / 83; FP32 59k hexes 102 / 86 / 82.
// Of a launch's 8 us at 216 cells 1.3 are the first loads, 2.2 the gradients, 2 the fluxes, 2
// the update: chains of dependent instructions at one wavefront a SIMD.
template <typename S>
__global__ __launch_bounds__(kBlock) void k_stage(DevMesh<S> m, DevParams prm, StageArgs sa,
                                                  const Ctrl *__restrict__ ctrl, const V4<S> *__restrict__ st_in,
                                                  V4<S> *__restrict__ st_out, double4 *__restrict__ t0,
                                                  Acc<S> *__restrict__ t1, double *__restrict__ dtl,
                                                  const double *__restrict__ fbody, double *__restrict__ partials,
                                                  double *__restrict__ bmin) {
    static_assert(kOneKernelCells <= 64, "a wavefront has the block's cells");
    extern __shared__ double lds[];
    const int done = ctrl->done;
    const int blk = xcd_block(blockIdx.x, gridDim.x, 1);
    const int e0 = m.blk_item_off[blk], e1 = m.blk_item_off[blk + 1];
    const bool force = block_force(m, prm, blk);
    S *sF = reinterpret_cast<S *>(lds);
    float4 *rec = reinterpret_cast<float4 *>(reinterpret_cast<char *>(lds) + staged_offset<S>(m.max_items));
    DevPatch *sP = reinterpret_cast<DevPatch *>(rec + kLocalRec<S> * m.max_local);
    // a place's cell, neighbours and weights
    constexpr int kPer = 16 / sizeof(S), kPieces = (3 * kMaxSlots + kPer - 1) / kPer;
    int i = -1, nbr[kMaxSlots];
    float4 w[kPieces];
    auto place = [&](int k) {
        const int p = blk * m.max_local + k;
        i = k < m.max_local ? m.loc_cell[p] : -1;
        if (k < m.max_local) {
#pragma unroll
            for (int s = 0; s < kMaxSlots; s++) nbr[s] = s < m.max_slots ? m.loc_nbr[s * m.n_places + p] : kNoNbr;
#pragma unroll
            for (int q = 0; q < kPieces; q++)
                if (q * kPer < 3 * m.max_slots) w[q] = m.loc_w[(size_t)q * m.n_places + p];
        }
    };
    place(threadIdx.x);
    for (int k = threadIdx.x; k < m.n_patches; k += kBlock) sP[k] = m.patches[k];
    const int e = e0 + threadIdx.x;
    Item<S> it{};
    uint32_t places = 0;
    if (e < e1) {
        it = load_item<S>(m, e);
        places = m.it_loc[e];
    }
    const int c = blk * m.block_cells + threadIdx.x;
    const bool live = (int)threadIdx.x < m.block_cells && c < m.N;
    CellIn<S> in;
    if (live) {
        in.faces = load_faces<S, true>(m, c);
        load_rk<S, true>(m, sa, force, c, t0, t1, dtl, fbody, in);
    }
    if (done) return;
    __syncthreads();
    DevMesh<S> ml = m;
    ml.patches = sP;
    for (int k = threadIdx.x; k < m.max_local; k += kBlock) {
        if (k != (int)threadIdx.x) place(k);
        if (i < 0) break;
        S g[12];
        const auto weight = [&](int s, int c) {
            const int q = 3 * s + c;
            S v[kPer];
            __builtin_memcpy(v, &w[q / kPer], 16);
            return v[q % kPer];
        };
        lsq_sums<S, kMaxSlots>(ml, i, nbr, kMaxSlots, weight, GlobalStates<S, Rec1>{st_in, Rec1{}}, g);
        LocalLoader<S>::put(rec + kLocalRec<S> * k, st_in[i], g);
    }
    __syncthreads();
    for (int f = e; f < e1; f += kBlock) {
        if (f != e) {
            it = load_item<S>(m, f);
            places = m.it_loc[f];
        }
        S F[4];
        item_flux<S>(ml, prm, it, LocalLoader<S>{rec, places}, prm.visc3_invgam, INFINITY, F);
#pragma unroll
        for (int q = 0; q < 4; q++) sF[q * m.max_items + (f - e0)] = F[q];
    }
    __syncthreads();
    double sq[4] = {0, 0, 0, 0};
    double dt = 1e300;
    const int err = live ? cell_update<S, true>(m, prm, sa, sF, force, c, in, st_out, t0, t1, dtl, sq, dt) : 0;
    block_sums(sa, blk, sq, err, partials);
    // the block's cells are the first wavefront's
    if (bmin && threadIdx.x < 64) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) dt = fmin(dt, __shfl_xor(dt, off, 64));
        if (threadIdx.x == 0) bmin[blk] = dt;
    }
}

// Global minimum of the local time steps for the "min" and "talts" modes
// (Solver.cpp:1746-1773): the blocks' minima, by this kernel or by k_stage, then
// k_dt_apply.
__global__ __launch_bounds__(kBlock) void k_dt_blockmin(int N, const Ctrl *__restrict__ ctrl,
                                                        const double *__restrict__ dtl, double *__restrict__ bmin) {
    if (ctrl->done) return;
    __shared__ double red[kBlock / 64];
    const int i = blockIdx.x * kBlock + threadIdx.x;
    double v = (i < N) ? dtl[i] : 1e300;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmin(v, __shfl_xor(v, off, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = red[0];
        for (int q = 1; q < kBlock / 64; q++) s = fmin(s, red[q]);
        bmin[blockIdx.x] = s;
    }
}

// Every block takes the minimum over all blocks' minima: by its whole width (by one
// thread, one after the other, 6.4 us at 64 blocks; step of 16k cells 57 -> 52 us).
__global__ __launch_bounds__(kBlock) void k_dt_apply(int N, int nblk, int mode, const Ctrl *__restrict__ ctrl,
                                                     const double *__restrict__ bmin, double *__restrict__ dtl) {
    if (ctrl->done) return;
    __shared__ double red[kBlock / 64];
    double s = 100000000000.0;
    for (int q = threadIdx.x; q < nblk; q += kBlock) s = (bmin[q] < s) ? bmin[q] : s;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s = fmin(s, __shfl_xor(s, off, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    double smin = red[0];
#pragma unroll
    for (int q = 1; q < kBlock / 64; q++) smin = fmin(smin, red[q]);
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= N) return;
    const double mn = smin;
    if (mode == PLBFS_DT_MIN) dtl[i] = mn;
    else dtl[i] = mn * pow(2.0, floor(log2(dtl[i] / mn)));
}

template <typename S>
__global__ __launch_bounds__(kBlock) void k_init_dt(int N, DevParams prm, const Ctrl *__restrict__ ctrl,
                                                    const double *__restrict__ cfl_area,
                                                    const double *__restrict__ vol, const V4<S> *__restrict__ st,
                                                    double *__restrict__ dtl) {
    if (ctrl->done) return;
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= N) return;
    const double r0 = std::is_same<S, float>::value ? prm.rho0 : 0.0;
    if (prm.time_stepping == PLBFS_DT_CONSTANT) dtl[i] = prm.cfl;
    else dtl[i] = local_dt(prm, prm.visc, r0 + (double)st[i].x, (double)st[i].y, cfl_area[i], vol[i]);
}

__global__ __launch_bounds__(kFinalizeThreads) void k_finalize(int nblk, double n_cells, double ref_rho,
                                                               double ref_mom, double tol, int stop_on_rebuild,
                                                               Ctrl *__restrict__ ctrl,
                                                               const double *__restrict__ partials,
                                                               double *__restrict__ hist, int hist_cap) {
    if (ctrl->done) return;
    __shared__ double red[kFinalizeThreads][5];
    double s[5] = {0, 0, 0, 0, 0};
    // a thread's partials b = tid, tid + T, ... in that order; four at a time
    // with all their loads issued before the sums
    constexpr int kU = 4;
    for (int b0 = threadIdx.x; b0 < nblk; b0 += kFinalizeThreads * kU) {
        double v[kU][5];
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const int b = b0 + u * kFinalizeThreads;
            if (b < nblk)
                for (int c = 0; c < 5; c++) v[u][c] = partials[(size_t)b * 5 + c];
        }
#pragma unroll
        for (int u = 0; u < kU; u++) {
            if (b0 + u * kFinalizeThreads < nblk) {
                for (int c = 0; c < 4; c++) s[c] += v[u][c];
                s[4] = fmax(s[4], v[u][4]);
            }
        }
    }
    for (int c = 0; c < 5; c++) red[threadIdx.x][c] = s[c];
    __syncthreads();
    for (int off = kFinalizeThreads / 2; off > 0; off >>= 1) {
        if (threadIdx.x < off) {
            for (int c = 0; c < 4; c++) red[threadIdx.x][c] += red[threadIdx.x + off][c];
            red[threadIdx.x][4] = fmax(red[threadIdx.x][4], red[threadIdx.x + off][4]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const int step = ctrl->step;
        double r[4];
        r[0] = sqrt(red[0][0] / n_cells) / ref_rho;
        for (int c = 1; c < 4; c++) r[c] = sqrt(red[0][c] / n_cells) / ref_mom;
        for (int c = 0; c < 4; c++) ctrl->res[c] = r[c];
        if (step < hist_cap)
            for (int c = 0; c < 4; c++) hist[(size_t)step * 4 + c] = r[c];
        ctrl->step = step + 1;
        const int e = (int)red[0][4];
        if (e == 1) {
            ctrl->status = PLBFS_ERR_NAN;
            ctrl->done = 1;
        } else if (e == 2) {
            ctrl->status = PLBFS_ERR_RHO;
            ctrl->done = 1;
        } else {
            const double me = fmax(fmax(r[3], r[1]), r[2]);
            if (me < tol) {
                ctrl->converged = 1;
                ctrl->done = 1;
            }
        }
        // immersed nodes asked for new candidate lists: the host builds them
        // and continues with the next step
        if (stop_on_rebuild && ctrl->rebuild) ctrl->done = 1;
    }
}

// Cell records to [4][N] in file order; divide: conservatives to primitives.
__global__ __launch_bounds__(kBlock) void k_export(int N, const int32_t *__restrict__ inv,
                                                   const double4 *__restrict__ src, int divide,
                                                   double *__restrict__ out) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= N) return;
    const double4 q = src[inv[i]];
    out[i] = q.x;
    out[(size_t)N + i] = divide ? q.y / q.x : q.y;
    out[2 * (size_t)N + i] = divide ? q.z / q.x : q.z;
    out[3 * (size_t)N + i] = divide ? q.w / q.x : q.w;
}

// One residual evaluation for diagnostics: flux gather only (stage-independent).
template <typename S>
__global__ __launch_bounds__(kBlock) void k_residual_only(DevMesh<S> m, DevParams prm,
                                                          const V4<S> *__restrict__ st_in,
                                                          const V4<S> *__restrict__ grad,
                                                          const double *__restrict__ fbody,
                                                          double *__restrict__ Rout) {
    extern __shared__ double lds[];
    const int N = m.N;
    const int blk = xcd_block(blockIdx.x, gridDim.x, m.xcd_remap);
    const int nslot = m.max_items;
    const S *sF = reinterpret_cast<const S *>(lds);
    if (m.stage) block_fluxes<S, true>(m, prm, st_in, grad, lds, blk);
    else block_fluxes<S, false>(m, prm, st_in, grad, lds, blk);
    __syncthreads();
    const int c_end = min(N, (blk + 1) * m.block_cells);
    for (int i = blk * m.block_cells + threadIdx.x; i < c_end; i += kBlock) {
        double R[4];
        gather_residual<S>(m, i, load_faces<S>(m, i), sF, nslot, 1, 0, R);
        if (prm.use_body_force) {
            R[1] += fbody[i];
            R[2] += fbody[(size_t)N + i];
            R[3] += fbody[2 * (size_t)N + i];
        }
        for (int q = 0; q < 4; q++) Rout[(size_t)q * N + i] = R[q];
    }
}

}  // namespace

// ---------------------------------------------------------------------------
// Context
// ---------------------------------------------------------------------------

// ---- the time loop without allocation --------------------------------------
// plbfs_run_noalloc works in this array instead of the context's control block,
// partials, dt minima and history; it allocates nothing, builds no graph and
// creates no events.  Each device holds its own copy until the process ends;
// kScratchBytes bounds what one call may use.  Calls that overlap on one
// device share the array and race.
constexpr size_t kScratchBytes = (size_t)8 << 20;
// The bound counts kFluxBlockCells cells a block where the mesh size chose the block
// size; the partials of the smaller blocks it may choose (up to 1,024 blocks instead of 256,
// 40 B each and 8 B for a minimum) fit behind it.
constexpr size_t kScratchSpare = (size_t)40 << 10;
static_assert(48 * (kResidentBlocks - 256) + 512 <= kScratchSpare, "partials and minima of the smallest blocks fit");
static __device__ __align__(256) double scratch[(kScratchBytes + kScratchSpare) / sizeof(double)];

constexpr int kMaxScratchDevices = 64;
static std::mutex g_scratch_mu;
static char *g_scratch_ptr[kMaxScratchDevices];

// This device's address of the scratch array; called by create_ctx with the
// context's device current, once per device.
static int resolve_scratch(int device, char **out) {
    if (device < 0 || device >= kMaxScratchDevices)
        return plbfs_fail(PLBFS_ERR_HIP, "device %d: scratch table holds %d devices", device, kMaxScratchDevices);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        void *p = nullptr;
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return plbfs_fail(PLBFS_ERR_HIP, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
        g_scratch_ptr[device] = static_cast<char *>(p);
    }
    *out = g_scratch_ptr[device];
    return PLBFS_OK;
}

void drop_graphs(plbfs_ctx *c) {
    for (hipGraphExec_t *g : {&c->graph_exec, &c->graph_many}) {
        if (*g) (void)hipGraphExecDestroy(*g);
        *g = nullptr;
    }
}

static int release(plbfs_ctx *c) {
    drop_graphs(c);
    for (void *p : c->allocs) hipFree(p);
    c->allocs.clear();
    for (void *p : c->ibm_allocs) hipFree(p);
    c->ibm_allocs.clear();
    for (hipEvent_t *e : {&c->ev0, &c->ev1}) {
        if (*e) (void)hipEventDestroy(*e);
        *e = nullptr;
    }
    if (c->host) (void)hipHostFree(c->host);
    c->host = nullptr;
    if (c->stream) {
        hipStreamDestroy(c->stream);
        c->stream = nullptr;
    }
    return PLBFS_OK;
}

extern "C" int plbfs_device_count(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

static bool env_flag(const char *name, bool def) {
    const char *v = std::getenv(name);
    if (!v || !v[0]) return def;
    return v[0] != '0';
}

extern "C" int plbfs_create(const plbfs_mesh_view *mesh, const plbfs_params *params, const plbfs_patch *patches,
                            int32_t n_patches, const int32_t *bface_patch, plbfs_ctx **out) {
    // cells per flux block (a multiple of 64), by default chosen for the mesh
    const char *bc = std::getenv("PLBFS_BLOCK_CELLS");
    const int block_cells = bc ? std::atoi(bc) : 0;
    if (bc && (block_cells < 64 || block_cells % 64 || block_cells > 4 * kBlock))
        return plbfs_fail(PLBFS_ERR_INPUT, "PLBFS_BLOCK_CELLS must be a multiple of 64 up to %d", 4 * kBlock);
    // measured on MI355X (4.09M tets): staging the flux block's own records in
    // LDS costs more (staging phase + barrier) than the L2 traffic it saves,
    // while staging the gradient kernel's 256 states saves 12 %; flux staging
    // is therefore opt-in (PLBFS_FLUX_STAGE=1) and gradient staging opt-out
    const bool flux_stage = env_flag("PLBFS_FLUX_STAGE", false);
    // faces between two blocks: both blocks evaluate them, or, with
    // PLBFS_SPLIT_BORDER=1, a separate border pass evaluates each once.
    // Measured on MI355X (4.09M tets): the border pass makes the flux step
    // slower (FP64 0.555 -> 0.617 ms, FP32 0.331 -> 0.364 ms; its faces
    // gather both sides from global memory), so duplication is the default
    const bool split = env_flag("PLBFS_SPLIT_BORDER", false);
    const int rc = create_ctx(mesh, params, patches, n_patches, bface_patch, block_cells, 1, flux_stage, split, out);
    if (rc == PLBFS_OK && !bc) (*out)->bound_blocks = (mesh->n_cells + kFluxBlockCells - 1) / kFluxBlockCells;
    return rc;
}

// Fixed ghost states to the device: (rho, u, v, w) per boundary face in the
// storage precision (FP32: rho as the deviation from rho0).
static int upload_ghost_fixed(plbfs_ctx *c) {
    const size_t G = (size_t)c->L.G;
    if (G == 0) return PLBFS_OK;
    if (!c->f32) {
        HIP_TRY(hipMemcpy(c->b_fix, c->ghost_fixed.data(), G * 4 * sizeof(double), hipMemcpyHostToDevice));
    } else {
        std::vector<float> h(G * 4);
        for (size_t k = 0; k < G * 4; k++)
            h[k] = (float)(c->ghost_fixed[k] - ((k & 3) == 0 ? c->prm.rho0 : 0.0));
        HIP_TRY(hipMemcpy(c->b_fix, h.data(), h.size() * sizeof(float), hipMemcpyHostToDevice));
    }
    return PLBFS_OK;
}

int create_ctx(const plbfs_mesh_view *mesh, const plbfs_params *params, const plbfs_patch *patches,
               int32_t n_patches, const int32_t *bface_patch, int block_cells, int lds_cases, bool flux_stage,
               bool split_border, plbfs_ctx **out) {
    if (!mesh || !params || !out) return plbfs_fail(PLBFS_ERR_INPUT, "null argument");
    *out = nullptr;
    const plbfs_params &p = *params;
    if (!(p.visc > 0) || !(p.gamma > 0) || !(p.cfl > 0) || !(p.max_velocity > 0) || !(p.ref_rho > 0))
        return plbfs_fail(PLBFS_ERR_INPUT, "visc, gamma, cfl, max_velocity and ref_rho must be positive");
    if (p.time_stepping < 0 || p.time_stepping > 3 || p.gradient_type < 0 || p.gradient_type > 2)
        return plbfs_fail(PLBFS_ERR_INPUT, "bad time_stepping or gradient_type");
    if (p.precision != PLBFS_FP64 && p.precision != PLBFS_FP32)
        return plbfs_fail(PLBFS_ERR_INPUT, "bad precision %d", p.precision);
    if (plbfs_device_count() <= 0) return plbfs_fail(PLBFS_ERR_NODEVICE, "no HIP device visible");
    auto *c = new plbfs_ctx();
    c->params = p;
    c->f32 = p.precision == PLBFS_FP32;
    c->patches.assign(patches, patches + n_patches);
    int rc = build_layout(*mesh, p, patches, n_patches, bface_patch, block_cells, split_border, c->L);
    if (rc) {
        delete c;
        return rc;
    }
    const Layout &L = c->L;
    const size_t sbytes = c->f32 ? sizeof(float) : sizeof(double);
    const bool stage = flux_stage;
    c->lds_bytes = lds_cases == 1
                       ? (c->f32 ? flux_lds_bytes<float>(L.max_items_per_block, L.block_cells, stage)
                                 : flux_lds_bytes<double>(L.max_items_per_block, L.block_cells, stage))
                       : (size_t)L.max_items_per_block * 4 * sbytes * lds_cases;
    if (c->lds_bytes > kMaxLds) {
        // L refers into c: read what the message needs before c is freed
        const size_t need = c->lds_bytes;
        const int slots = L.max_items_per_block;
        delete c;
        return plbfs_fail(PLBFS_ERR_INPUT, "a block needs %zu B of LDS for %d face slots x %d cases (limit %d B)",
                          need, slots, lds_cases, kMaxLds);
    }
    auto fail = [&](int r) {
        release(c);
        delete c;
        return r;
    };
    if (hipGetDevice(&c->device) != hipSuccess) return fail(plbfs_fail(PLBFS_ERR_HIP, "hipGetDevice"));
    if ((rc = resolve_scratch(c->device, &c->scratch))) return fail(rc);
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess)
        return fail(plbfs_fail(PLBFS_ERR_HIP, "hipStreamCreate"));
    if (hipEventCreate(&c->ev0) != hipSuccess || hipEventCreate(&c->ev1) != hipSuccess ||
        hipHostMalloc((void **)&c->host, kHostBytes, hipHostMallocDefault) != hipSuccess)
        return fail(plbfs_fail(PLBFS_ERR_HIP, "events and host buffer"));
    const int N = L.N;
    c->bound_blocks = L.n_blocks;
    // A stage in one kernel on meshes below 65,536 cells (blocks of 64 cells; larger blocks
    // do not fit).  The repeated gradients grow with the mesh, and the gain falls: 59k hexes in
    // FP64 118 -> 105 us a step, 64k tets 106 -> 83.
    if (L.one_kernel && lds_cases == 1 && !stage) {
        const size_t b = (c->f32 ? staged_offset<float>(L.max_items_per_block)
                                 : staged_offset<double>(L.max_items_per_block)) +
                         (size_t)L.max_local * 16 * (c->f32 ? kLocalRec<float> : kLocalRec<double>) + (size_t)n_patches * sizeof(DevPatch);
        if (b <= kMaxStageLds) c->stage_lds = b;
    }
    DevMesh<double> &d = c->dm;
    d.N = N;
    d.G = L.G;
    d.n_blocks = L.n_blocks;
    d.max_items = L.max_items_per_block;
    d.E = L.n_items;
    d.border0 = L.border0;
    d.n_border = (int)L.n_border;
    d.bflux = nullptr;
    d.blk_force = nullptr;
    d.max_slots = *std::max_element(L.st_cnt.begin(), L.st_cnt.end());
    for (int a = 0; a < 3; a++) d.b0[a] = L.b0[a];
    d.block_cells = L.block_cells;
    d.stage = stage ? 1 : 0;
    d.grad_stage = env_flag("PLBFS_GRAD_STAGE", true) ? 1 : 0;
    c->cell_grid = (N + kBlock - 1) / kBlock;
    // Consecutive blocks on one XCD keep the cells that they share in its L2.  k_grad and
    // k_stage always take that order (4.1M tets in FP32 125 -> 111 us a launch, 221k hexes in
    // FP64 16.1 -> 15.4, with the records then written where flux blocks of the same XCD read
    // them; step of 32k hexes 50.4 -> 47.4 us).  Flux blocks take it on meshes of up to
    // kXcdCells cells: step of 221k hexes in FP64 201.9 -> 190.6 us, of 681k 565 -> 559, FP32
    // 351.2 -> 349.4; 1.1M hexes in FP64 901 -> 925, 1.1M tets in FP32 475 -> 482 and 4.1M tets
    // in FP64 2.54 -> 2.65 ms: what the blocks of one XCD stream through its L2 then
    // drives the shared cells out.
    const char *nx = std::getenv("PLBFS_XCD_REMAP");
    d.xcd_remap = nx && nx[0] ? nx[0] == '1' : N <= kXcdCells;
    std::vector<DevPatch> dp(n_patches);
    for (int q = 0; q < n_patches; q++) {
        dp[q].rho_type = patches[q].rho_type;
        dp[q].vel_type = patches[q].vel_type;
        dp[q].is_empty = patches[q].is_empty;
        const bool keeps = rho_keeps_ghost(patches[q].rho_type) || vel_keeps_ghost(patches[q].vel_type);
        dp[q].flags = (patches[q].rho_type == 3 || patches[q].vel_type == 3 || keeps ? kGhostGradFromCell : 0) |
                      (keeps ? kGhostFixed : 0);
        dp[q].rho = patches[q].rho;
        dp[q].u = patches[q].u;
        dp[q].v = patches[q].v;
        dp[q].w = patches[q].w;
    }
    // the entries of the border pass hold indices beyond 16 bits; without it a slot
    // is below kMaxLds / 16
    static_assert(kMaxLds / 16 < kNoEnt >> 1, "slots fit the 16-bit entries");
    d.max_ent = 1;
    for (int i = 0; i < N; i++) d.max_ent = std::max(d.max_ent, L.g_off[i + 1] - L.g_off[i]);
    d.g_ent = nullptr;
    d.g_ent_split = nullptr;
    if (d.n_border > 0)
        rc = upload(c, (int32_t **)&d.g_ent_split,
                    entries_by_face<int32_t>(L, d.max_ent, -1, [](int32_t e) { return e; }));
    else
        rc = upload(c, (uint16_t **)&d.g_ent, entries_by_face<uint16_t>(L, d.max_ent, kNoEnt, [](int32_t e) {
                        return (uint16_t)((e >> 2) << 1 | (e & 1));
                    }));
    if (rc) return fail(rc);
    d.max_local = L.max_local;
    d.n_places = L.n_blocks * L.max_local;
    d.n_patches = n_patches;
    d.loc_cell = d.loc_nbr = nullptr;
    d.it_loc = nullptr;
    d.loc_w = nullptr;
    int32_t *loc_nbr = nullptr;
    float4 *loc_w = nullptr;
    if (c->stage_lds) {
        std::vector<int32_t> v(L.loc_cell);
        v.insert(v.end(), L.it_loc.begin(), L.it_loc.end());
        const size_t P = (size_t)d.n_places, per = 16 / sbytes;
        if ((rc = upload(c, (int32_t **)&d.loc_cell, v)) ||
            (rc = dalloc(c, (void **)&loc_nbr, P * kMaxSlots * sizeof(int32_t))) ||
            (rc = dalloc(c, (void **)&loc_w, P * ((3 * kMaxSlots + per - 1) / per) * sizeof(float4))))
            return fail(rc);
        d.it_loc = reinterpret_cast<const uint32_t *>(d.loc_cell + P);
        d.loc_nbr = loc_nbr;
        d.loc_w = loc_w;
    }
    // patches of the boundary faces, then their partners; at least one of each
    std::vector<int32_t> bface = L.b_patch;
    if (bface.empty()) bface.push_back(0);
    const size_t partners = bface.size();
    bface.insert(bface.end(), L.b_partner.begin(), L.b_partner.end());
    if (L.b_partner.empty()) bface.push_back(-1);
    std::vector<double> bdmag = L.b_dmag;
    if (bdmag.empty()) bdmag.push_back(1.0);
    c->ghost_fixed = L.b_fixed;
    c->ghost_state_set = !L.needs_ghost_state;
    if ((rc = dalloc(c, (void **)&c->b_fix, (size_t)std::max(L.G, 1) * 4 * sbytes))) return fail(rc);
    d.b_fix = c->f32 ? nullptr : (const double4 *)c->b_fix;
    d.corr = nullptr;
    if ((rc = upload(c, (uint8_t **)&d.st_cnt, L.st_cnt)) || (rc = upload(c, (int32_t **)&d.st_nbr, L.st_nbr)) ||
        (rc = upload(c, (double **)&d.vol, L.vol)) || (rc = upload(c, (double **)&d.inv_vol, L.inv_vol)) ||
        (rc = upload(c, (double **)&d.cfl_area, L.cfl_area)) ||
        (rc = upload(c, (int32_t **)&d.blk_item_off, L.blk_item_off)) ||
        (rc = upload(c, (float4 **)&d.it_p, c->f32 ? pack_items<float>(L) : pack_items<double>(L))) ||
        (rc = upload(c, (uint16_t **)&d.it_side, std::vector<uint16_t>(L.it_side.begin(), L.it_side.end()))) ||
        (rc = upload(c, (int32_t **)&d.b_patch, bface)) || (rc = upload(c, (DevPatch **)&d.patches, dp)) ||
        (rc = upload(c, &c->inv, L.inv)))
        return fail(rc);
    d.b_partner = d.b_patch + partners;
    if (!c->f32) {
        std::vector<double> dt((size_t)L.n_items);
        for (size_t e = 0; e < dt.size(); e++) dt[e] = L.it_geo[kGeoPerItem * e + 4];
        if ((rc = upload(c, (double **)&d.st_w, L.st_w)) || (rc = upload(c, (double **)&d.it_dt, dt)) ||
            (rc = upload(c, (double **)&d.b_dmag, bdmag)))
            return fail(rc);
    } else {
        // FP32 storage: the same arrays rounded once from the FP64 precompute;
        // patch densities become deviations from rho0
        DevMesh<float> &e = c->dm32;
        e.N = d.N; e.G = d.G; e.n_blocks = d.n_blocks; e.max_items = d.max_items; e.E = d.E;
        e.border0 = d.border0; e.n_border = d.n_border; e.bflux = nullptr; e.blk_force = nullptr;
        e.xcd_remap = d.xcd_remap;
        for (int a = 0; a < 3; a++) e.b0[a] = (float)L.b0[a];
        e.block_cells = d.block_cells;
        e.stage = d.stage;
        e.grad_stage = d.grad_stage;
        e.max_slots = d.max_slots;
        e.st_cnt = d.st_cnt; e.st_nbr = d.st_nbr; e.vol = d.vol; e.inv_vol = d.inv_vol; e.cfl_area = d.cfl_area;
        e.blk_item_off = d.blk_item_off; e.it_p = d.it_p; e.it_side = d.it_side; e.it_dt = nullptr;
        e.g_ent = d.g_ent; e.g_ent_split = d.g_ent_split; e.max_ent = d.max_ent; e.b_patch = d.b_patch; e.b_partner = d.b_partner;
        e.b_fix = (const float4 *)c->b_fix;
        e.loc_cell = d.loc_cell; e.loc_nbr = d.loc_nbr; e.loc_w = d.loc_w; e.it_loc = d.it_loc;
        e.max_local = d.max_local; e.n_places = d.n_places; e.n_patches = d.n_patches;
        auto to32 = [](const std::vector<double> &v) { return std::vector<float>(v.begin(), v.end()); };
        std::vector<DevPatch> dp32 = dp;
        for (auto &q : dp32) q.rho -= p.ref_rho;
        if ((rc = upload(c, (float **)&e.st_w, to32(L.st_w))) ||
            (rc = upload(c, (float **)&e.b_dmag, to32(bdmag))) || (rc = upload(c, (float **)&e.corr, to32(L.corr))) ||
            (rc = upload(c, (DevPatch **)&e.patches, dp32)))
            return fail(rc);
    }
    if (c->stage_lds) {
        const dim3 grid((d.n_places + kBlock - 1) / kBlock);
        if (c->f32) hipLaunchKernelGGL(k_places<float>, grid, dim3(kBlock), 0, c->stream, c->dm32, loc_nbr, loc_w);
        else hipLaunchKernelGGL(k_places<double>, grid, dim3(kBlock), 0, c->stream, c->dm, loc_nbr, loc_w);
        if (hipGetLastError() != hipSuccess) return fail(plbfs_fail(PLBFS_ERR_HIP, "k_places"));
    }
    const size_t n4 = (size_t)4 * N * sbytes;
    const size_t nacc = (size_t)4 * N * (c->f32 ? sizeof(float) : sizeof(double));
    if ((rc = dalloc(c, (void **)&c->stA, n4)) || (rc = dalloc(c, (void **)&c->stB, (size_t)4 * N * sizeof(double))) ||
        (rc = dalloc(c, (void **)&c->t0, (size_t)4 * N * sizeof(double))) || (rc = dalloc(c, (void **)&c->t1, nacc)) ||
        (rc = dalloc(c, (void **)&c->grad, (size_t)4 * (c->f32 ? kGradRec<float> : kGradRec<double>) * N * sbytes)) ||
        (rc = dalloc(c, (void **)&c->dtl, (size_t)N * sizeof(double))) ||
        (rc = dalloc(c, (void **)&c->fbody, (size_t)3 * N * sizeof(double))) ||
        (rc = dalloc(c, (void **)&c->partials, (size_t)L.n_blocks * 5 * sizeof(double))) ||
        (rc = dalloc(c, (void **)&c->bmin, (size_t)c->n_min() * sizeof(double))) ||
        (rc = dalloc(c, (void **)&c->ctrl, sizeof(Ctrl))) ||
        (rc = dalloc(c, &c->bflux, (size_t)4 * std::max<int64_t>(L.n_border, 1) * sbytes)))
        return fail(rc);
    c->dm.bflux = (double *)c->bflux;
    c->dm32.bflux = (float *)c->bflux;
    if (hipMemsetAsync(c->fbody, 0, (size_t)3 * N * sizeof(double), c->stream) != hipSuccess ||
        hipMemsetAsync(c->ctrl, 0, sizeof(Ctrl), c->stream) != hipSuccess)
        return fail(plbfs_fail(PLBFS_ERR_HIP, "clear body force and control block"));
    DevParams &prm = c->prm;
    prm.visc = p.visc;
    prm.gamma = p.gamma;
    prm.invgam = 1.0 / p.gamma;
    prm.visc3_invgam = p.visc * 3 / p.gamma;
    prm.c45 = 4.5 * prm.invgam;
    prm.c15 = 1.5 * prm.invgam;
    prm.force = p.force;
    prm.cfl = p.cfl;
    prm.ceff = p.max_velocity * std::sqrt(1 - p.gamma + std::pow(p.gamma / std::sqrt(3) / p.max_velocity, 2));
    prm.ref_rho = p.ref_rho;
    prm.rho0 = p.ref_rho;
    prm.ref_mom = p.ref_rho * p.max_velocity;
    prm.tol = p.tolerance;
    prm.time_stepping = p.time_stepping;
    prm.use_body_force = 0;
    const char *g = std::getenv("PLBFS_NO_GRAPH");
    c->use_graph = !(g && g[0] == '1');
    if ((rc = upload_ghost_fixed(c))) return fail(rc);
    *out = c;
    return PLBFS_OK;
}

extern "C" int plbfs_destroy(plbfs_ctx *c) {
    if (!c) return PLBFS_OK;
    if (c->stream) hipStreamSynchronize(c->stream);
    release(c);
    delete c;
    return PLBFS_OK;
}

static int to_device_state(plbfs_ctx *c, const double *rho, const double *u, const double *v, const double *w,
                           double *dst) {
    const int N = c->L.N;
    std::vector<double> h((size_t)4 * N);  // cell records (rho,u,v,w), Hilbert order
    const double *src[4] = {rho, u, v, w};
    for (int n = 0; n < N; n++)
        for (int q = 0; q < 4; q++) h[(size_t)4 * n + q] = src[q][c->L.perm[n]];
    HIP_TRY(hipMemcpy(dst, h.data(), h.size() * sizeof(double), hipMemcpyHostToDevice));
    return PLBFS_OK;
}

int fields_to_host(plbfs_ctx *c, const double *src, double *const out[4]) {
    const size_t N = (size_t)c->L.N, bytes = N * sizeof(double);
    if (4 * bytes <= kHostBytes) {
        HIP_TRY(hipMemcpyAsync(c->host, src, 4 * bytes, hipMemcpyDeviceToHost, c->stream));
        HIP_TRY(hipStreamSynchronize(c->stream));
        for (int q = 0; q < 4; q++)
            if (out[q]) std::memcpy(out[q], c->host + q * bytes, bytes);
        return PLBFS_OK;
    }
    for (int q = 0; q < 4; q++)
        if (out[q]) HIP_TRY(hipMemcpyAsync(out[q], src + q * N, bytes, hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    return PLBFS_OK;
}

// Copies nf interleaved values per cell back to file order (one array per value).
static int from_device_fields(plbfs_ctx *c, const double *src, int nf, double *const *out) {
    const int N = c->L.N;
    std::vector<double> h((size_t)nf * N);
    HIP_TRY(hipMemcpy(h.data(), src, h.size() * sizeof(double), hipMemcpyDeviceToHost));
    for (int q = 0; q < nf; q++)
        if (out[q])
            for (int n = 0; n < N; n++) out[q][c->L.perm[n]] = h[(size_t)nf * n + q];
    return PLBFS_OK;
}

extern "C" int plbfs_set_state(plbfs_ctx *c, const double *rho, const double *u, const double *v, const double *w) {
    if (!c || !rho || !u || !v || !w) return plbfs_fail(PLBFS_ERR_INPUT, "null argument");
    // the conservative accumulator starts as a copy of the primitives (Solver.cpp:195)
    int rc = to_device_state(c, rho, u, v, w, c->t0);
    if (rc) return rc;
    const int N = c->L.N;
    if (!c->f32) {
        // on the stream that reads it: a copy inside the device need not block the host
        HIP_TRY(hipMemcpyAsync(c->stA, c->t0, (size_t)4 * N * sizeof(double), hipMemcpyDeviceToDevice, c->stream));
        HIP_TRY(hipStreamSynchronize(c->stream));
    } else {
        std::vector<float> h((size_t)4 * N);
        const double *src[4] = {rho, u, v, w};
        for (int n = 0; n < N; n++)
            for (int q = 0; q < 4; q++)
                h[(size_t)4 * n + q] = (float)(src[q][c->L.perm[n]] - (q == 0 ? c->prm.rho0 : 0.0));
        HIP_TRY(hipMemcpy(c->stA, h.data(), h.size() * sizeof(float), hipMemcpyHostToDevice));
    }
    c->total_steps = 0;
    return PLBFS_OK;
}

extern "C" int plbfs_set_ghost_state(plbfs_ctx *c, const double *rho, const double *u, const double *v,
                                     const double *w) {
    if (!c || !rho || !u || !v || !w) return plbfs_fail(PLBFS_ERR_INPUT, "null argument");
    // only the components the reference's ghost update leaves unwritten take
    // these values (src/Solution.cpp:759-833); the parabolic u, v stay
    for (int b = 0; b < c->L.G; b++) {
        const plbfs_patch &P = c->patches[c->L.b_patch[b]];
        double *q = &c->ghost_fixed[(size_t)4 * b];
        if (rho_keeps_ghost(P.rho_type)) q[0] = rho[b];
        if (P.vel_type == 7 || P.vel_type == 9) {
            q[1] = u[b];
            q[2] = v[b];
        }
        if (vel_keeps_ghost(P.vel_type)) q[3] = w[b];
    }
    HIP_TRY(hipStreamSynchronize(c->stream));
    int rc = upload_ghost_fixed(c);
    if (rc) return rc;
    c->ghost_state_set = true;
    return PLBFS_OK;
}

// Refuses to advance a context whose patches keep initial ghost values that
// were never given.
static int check_ghost_state(const plbfs_ctx *c) {
    if (c->ghost_state_set) return PLBFS_OK;
    return plbfs_fail(PLBFS_ERR_INPUT,
                      "a patch keeps the ghost's initial state (density 4, 5, 9 or velocity 4, 5, 7, 9): "
                      "call plbfs_set_ghost_state first");
}

extern "C" int plbfs_get_state(plbfs_ctx *c, double *rho, double *u, double *v, double *w) {
    if (!c) return plbfs_fail(PLBFS_ERR_INPUT, "null argument");
    // FP32 storage: the FP64 conservative state t0 holds the solution (before
    // any step it still holds the initial primitives)
    double *outs[4] = {rho, u, v, w};
    double *tmp = c->stB;  // rewritten before it is read in a step
    hipLaunchKernelGGL(k_export, dim3((c->L.N + kBlock - 1) / kBlock), dim3(kBlock), 0, c->stream, c->L.N, c->inv,
                       (const double4 *)(c->f32 ? c->t0 : c->stA), c->f32 && c->total_steps > 0 ? 1 : 0, tmp);
    HIP_TRY(hipGetLastError());
    return fields_to_host(c, tmp, outs);
}

// ---- launches -------------------------------------------------------------

static void resolve_timing(plbfs_ctx *c) {
    for (auto &p : c->pending) {
        hipEventSynchronize(p.b);
        float ms = 0;
        hipEventElapsedTime(&ms, p.a, p.b);
        c->kstat[p.which].ms += ms;
        c->kstat[p.which].launches++;
        hipEventDestroy(p.a);
        hipEventDestroy(p.b);
    }
    c->pending.clear();
}

static const double kAlpha[4] = {1.0, 0.5, 0.5, 1.0};
static const double kBeta[4] = {1.0 / 6.0, 1.0 / 3.0, 1.0 / 3.0, 1.0 / 6.0};

// Device memory a time loop works in besides the context's fields: the control
// block, per-block residual partials, per-block dt minima and the residual
// history.  plbfs_run uses the context's own arrays, plbfs_run_noalloc carves
// them out of the file-scope scratch array.
struct RunScratch {
    Ctrl *ctrl;
    double *partials;  // [n_blocks * 5]
    double *bmin;      // [n_min()]
    double *hist;      // [hist_cap * 4]
    int hist_cap;
};

static RunScratch ctx_scratch(plbfs_ctx *c) { return RunScratch{c->ctrl, c->partials, c->bmin, c->hist, c->hist_cap}; }

static bool global_dt(const plbfs_ctx *c) {
    return c->params.time_stepping == PLBFS_DT_MIN || c->params.time_stepping == PLBFS_DT_TALTS;
}

// have_min: k_stage left its blocks' minima (a launch of k_dt_blockmin less: step of 16k
// cells 50.9 -> 49.1 us).
static void launch_dt_modes(plbfs_ctx *c, const RunScratch &w, bool have_min) {
    const int N = c->L.N, nb = c->cell_grid;
    if (global_dt(c)) {
        if (!have_min)
            hipLaunchKernelGGL(k_dt_blockmin, dim3(nb), dim3(kBlock), 0, c->stream, N, w.ctrl, c->dtl, w.bmin);
        hipLaunchKernelGGL(k_dt_apply, dim3(nb), dim3(kBlock), 0, c->stream, N, have_min ? c->L.n_blocks : nb,
                           c->params.time_stepping, w.ctrl, w.bmin, c->dtl);
    }
}

template <typename S>
static void launch_stages(plbfs_ctx *c, const DevMesh<S> &dm, const RunScratch &w, bool timed) {
    const int nb = c->L.n_blocks;
    void *in = c->stA, *outb = c->stB;
    for (int k = 0; k < 4; k++) {
        if (c->stage_lds) {
            const StageArgs sa{kAlpha[k], kBeta[k], k};
            TimedLaunch t(c, PLBFS_KSTAT_FLUX, timed);
            hipLaunchKernelGGL(k_stage<S>, dim3(nb), dim3(kBlock), c->stage_lds, c->stream, dm, c->prm, sa, w.ctrl,
                               (const V4<S> *)in, (V4<S> *)outb, (double4 *)c->t0, (Acc<S> *)c->t1, c->dtl, c->fbody,
                               w.partials, k == 3 && global_dt(c) ? w.bmin : nullptr);
            std::swap(in, outb);
            continue;
        }
        {
            TimedLaunch t(c, PLBFS_KSTAT_GRAD, timed);
            hipLaunchKernelGGL(k_grad<S>, dim3(c->cell_grid), dim3(kBlock), 0, c->stream, dm, w.ctrl, (const V4<S> *)in,
                               (V4<S> *)c->grad);
        }
        StageArgs sa{kAlpha[k], kBeta[k], k};
        {
            TimedLaunch t(c, PLBFS_KSTAT_FLUX, timed);
            if (dm.n_border > 0)
                hipLaunchKernelGGL(k_flux_border<S>, dim3((dm.n_border + kBlock - 1) / kBlock), dim3(kBlock), 0,
                                   c->stream, dm, c->prm, w.ctrl, (const V4<S> *)in, (const V4<S> *)c->grad);
            hipLaunchKernelGGL((dm.stage ? k_flux_update<S, true> : k_flux_update<S, false>), dim3(nb), dim3(kBlock),
                               c->lds_bytes, c->stream, dm, c->prm, sa, w.ctrl, (const V4<S> *)in,
                               (const V4<S> *)c->grad, (V4<S> *)outb, (double4 *)c->t0, (Acc<S> *)c->t1, c->dtl,
                               c->fbody, w.partials);
        }
        std::swap(in, outb);
    }
}

template <typename S>
static void launch_init_dt(plbfs_ctx *c, const DevMesh<S> &dm, const Ctrl *ctrl) {
    hipLaunchKernelGGL(k_init_dt<S>, dim3(c->cell_grid), dim3(kBlock), 0, c->stream, c->L.N, c->prm, ctrl,
                       dm.cfl_area, dm.vol, (const V4<S> *)c->stA, c->dtl);
}

// The loop's first launches: the local time steps of the current state.
static int launch_run_start(plbfs_ctx *c, const RunScratch &w) {
    if (c->f32) launch_init_dt<float>(c, c->dm32, w.ctrl);
    else launch_init_dt<double>(c, c->dm, w.ctrl);
    launch_dt_modes(c, w, false);
    HIP_TRY(hipGetLastError());
    return PLBFS_OK;
}

// rebuild: immersed nodes that drift half their list margin end the step
// replay so that the host rebuilds the lists (plbfs_run); without it they run
// on to the margin (plbfs_run_noalloc, which cannot allocate new lists).
static int launch_step(plbfs_ctx *c, const RunScratch &w, bool timed, bool rebuild) {
    const int nb = c->L.n_blocks;
    int rc = ibm_launch(c, w.ctrl, timed, rebuild);  // once per step, before the stages (Solver_gpu.cu:687-718)
    if (rc) return rc;
    if (c->f32) launch_stages<float>(c, c->dm32, w, timed);
    else launch_stages<double>(c, c->dm, w, timed);
    launch_dt_modes(c, w, c->stage_lds != 0);
    {
        TimedLaunch t(c, PLBFS_KSTAT_REDUCE, timed);
        hipLaunchKernelGGL(k_finalize, dim3(1), dim3(kFinalizeThreads), 0, c->stream, nb, (double)c->L.N,
                           c->prm.ref_rho, c->prm.ref_mom, c->prm.tol, rebuild ? 1 : 0, w.ctrl, w.partials,
                           w.hist, w.hist_cap);
    }
    HIP_TRY(hipGetLastError());
    return PLBFS_OK;
}

__global__ void k_clear_ctrl(Ctrl *ctrl) {
    if (threadIdx.x == 0) *ctrl = Ctrl{};
}

static int ensure_hist(plbfs_ctx *c, int steps) {
    if (steps <= c->hist_cap) return PLBFS_OK;
    drop_graphs(c);
    int cap = std::max(steps, 1024);
    int rc = dalloc(c, (void **)&c->hist, (size_t)cap * 4 * sizeof(double));
    if (rc) return rc;
    c->hist_cap = cap;
    return PLBFS_OK;
}

// Captures `steps` time steps into *exec unless that is done already.
static int build_graph(plbfs_ctx *c, int steps, hipGraphExec_t *exec) {
    if (*exec) return PLBFS_OK;
    hipGraph_t g;
    HIP_TRY(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
    int rc = PLBFS_OK;
    for (int s = 0; s < steps && rc == PLBFS_OK; s++) rc = launch_step(c, ctx_scratch(c), false, true);
    hipError_t e = hipStreamEndCapture(c->stream, &g);
    if (rc) return rc;
    if (e != hipSuccess) return plbfs_fail(PLBFS_ERR_HIP, "graph capture: %s", hipGetErrorString(e));
    e = hipGraphInstantiate(exec, g, nullptr, nullptr, 0);
    hipGraphDestroy(g);
    if (e != hipSuccess) {
        *exec = nullptr;
        return plbfs_fail(PLBFS_ERR_HIP, "graph instantiate: %s", hipGetErrorString(e));
    }
    return PLBFS_OK;
}

static void fill_result(plbfs_ctx *c, const Ctrl &h, float ms, plbfs_result *out) {
    c->total_steps += h.step;
    if (!out) return;
    out->status = h.status;
    out->steps = h.step;
    out->converged = h.converged;
    out->total_steps = c->total_steps;
    for (int q = 0; q < 4; q++) out->residual[q] = h.res[q];
    out->solve_ms = ms;
}

extern "C" int plbfs_run(plbfs_ctx *c, int32_t max_steps, plbfs_result *out) {
    if (!c || max_steps < 0) return plbfs_fail(PLBFS_ERR_INPUT, "bad arguments");
    int rc = check_ghost_state(c);
    if (rc) return rc;
    if ((rc = ensure_hist(c, max_steps))) return rc;
    const RunScratch w = ctx_scratch(c);
    hipLaunchKernelGGL(k_clear_ctrl, dim3(1), dim3(64), 0, c->stream, c->ctrl);
    if ((rc = launch_run_start(c, w))) return rc;
    const int interval = std::max(1, c->params.check_interval);
    const bool graph = c->use_graph && !c->timing;
    // the control block comes to the pinned buffer, with the history behind it
    // at the last check where it fits
    Ctrl h{};
    const size_t hist0 = 256, hist_bytes = (size_t)max_steps * 4 * sizeof(double);
    static_assert(sizeof(Ctrl) <= 256, "the history follows the control block");
    const bool small = hist0 + hist_bytes <= kHostBytes;
    bool have_hist = max_steps == 0;
    const GraphNeeds need(max_steps, interval);
    if (graph && ((need.many && (rc = build_graph(c, kGraphSteps, &c->graph_many))) ||
                  (need.one && (rc = build_graph(c, 1, &c->graph_exec)))))
        return rc;
    HIP_TRY(hipEventRecord(c->ev0, c->stream));
    for (int s = 0; s < max_steps;) {
        const int left = std::min(interval - s % interval, max_steps - s);  // steps to the next check
        int n = 1;
        if (graph && left >= kGraphSteps) {
            n = kGraphSteps;
            if ((rc = build_graph(c, n, &c->graph_many))) return rc;
            HIP_TRY(hipGraphLaunch(c->graph_many, c->stream));
        } else if (graph) {
            if ((rc = build_graph(c, 1, &c->graph_exec))) return rc;
            HIP_TRY(hipGraphLaunch(c->graph_exec, c->stream));
        } else if ((rc = launch_step(c, w, c->timing, true))) {
            return rc;
        }
        s += n;
        if (n == left) {
            have_hist = small && s == max_steps;
            HIP_TRY(hipEventRecord(c->ev1, c->stream));
            HIP_TRY(hipMemcpyAsync(c->host, c->ctrl, sizeof(Ctrl), hipMemcpyDeviceToHost, c->stream));
            if (have_hist)
                HIP_TRY(hipMemcpyAsync(c->host + hist0, c->hist, hist_bytes, hipMemcpyDeviceToHost, c->stream));
            HIP_TRY(hipStreamSynchronize(c->stream));
            std::memcpy(&h, c->host, sizeof h);
            if (h.done && h.rebuild && h.status == PLBFS_OK && !h.converged) {
                // new candidate lists around the nodes' positions after step
                // h.step, then on from there: the launches after the stop were
                // no-ops, so the loop resumes at the step count
                if ((rc = ibm_rebuild(c)) || (rc = ensure_hist(c, max_steps))) return rc;
                h.done = 0;
                h.rebuild = 0;
                HIP_TRY(hipMemcpyAsync(c->ctrl, &h, sizeof(Ctrl), hipMemcpyHostToDevice, c->stream));
                s = h.step;
                continue;
            }
            if (h.done) break;
        }
    }
    if (max_steps == 0) HIP_TRY(hipEventRecord(c->ev1, c->stream));
    HIP_TRY(hipEventSynchronize(c->ev1));
    resolve_timing(c);
    float ms = 0;
    hipEventElapsedTime(&ms, c->ev0, c->ev1);
    c->last_hist.assign((size_t)h.step * 4, 0.0);
    const size_t got = (size_t)std::min(h.step, c->hist_cap) * 4 * sizeof(double);
    if (have_hist) std::memcpy(c->last_hist.data(), c->host + hist0, got);
    else if (h.step > 0) HIP_TRY(hipMemcpy(c->last_hist.data(), c->hist, got, hipMemcpyDeviceToHost));
    fill_result(c, h, ms, out);
    return h.status;
}

static size_t round256(size_t b) { return (b + 255) / 256 * 256; }

// Bytes of scratch a run of max_steps steps needs on context c, as the bound counts them.
static size_t scratch_need(const plbfs_ctx *c, int64_t max_steps) {
    return round256(sizeof(Ctrl)) + round256((size_t)c->bound_blocks * 5 * sizeof(double)) +
           round256((size_t)c->cell_grid * sizeof(double)) + (size_t)max_steps * 4 * sizeof(double);
}

extern "C" int plbfs_run_noalloc(plbfs_ctx *c, int32_t max_steps, plbfs_result *out, double *hist_out) {
    if (!c || max_steps < 0) return plbfs_fail(PLBFS_ERR_INPUT, "bad arguments");
    if (!c->scratch) return plbfs_fail(PLBFS_ERR_HIP, "no scratch address for this context's device");
    if (int e = check_ghost_state(c)) return e;
    const size_t need = scratch_need(c, max_steps);
    if (need > kScratchBytes)
        return plbfs_fail(PLBFS_ERR_INPUT,
                          "plbfs_run_noalloc: %d cells in %d blocks and %d steps need %zu B of scratch, limit %zu B",
                          c->L.N, c->L.n_blocks, max_steps, need, kScratchBytes);
    char *p = c->scratch;
    RunScratch w;
    w.ctrl = reinterpret_cast<Ctrl *>(p);
    p += round256(sizeof(Ctrl));
    w.partials = reinterpret_cast<double *>(p);
    p += round256((size_t)c->L.n_blocks * 5 * sizeof(double));
    w.bmin = reinterpret_cast<double *>(p);
    p += round256((size_t)c->n_min() * sizeof(double));
    w.hist = reinterpret_cast<double *>(p);
    w.hist_cap = max_steps;
    const auto t0 = std::chrono::steady_clock::now();
    hipLaunchKernelGGL(k_clear_ctrl, dim3(1), dim3(64), 0, c->stream, w.ctrl);
    int rc = launch_run_start(c, w);
    if (rc) return rc;
    const int interval = std::max(1, c->params.check_interval);
    Ctrl h{};
    for (int s = 0; s < max_steps; s++) {
        if ((rc = launch_step(c, w, false, false))) return rc;
        if ((s + 1) % interval == 0 || s == max_steps - 1) {
            HIP_TRY(hipMemcpyAsync(c->host, w.ctrl, sizeof(Ctrl), hipMemcpyDeviceToHost, c->stream));
            HIP_TRY(hipStreamSynchronize(c->stream));
            std::memcpy(&h, c->host, sizeof h);
            if (h.done) break;
        }
    }
    if (max_steps == 0) HIP_TRY(hipStreamSynchronize(c->stream));
    const double ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    if (hist_out && h.step > 0)
        HIP_TRY(hipMemcpy(hist_out, w.hist, (size_t)h.step * 4 * sizeof(double), hipMemcpyDeviceToHost));
    c->last_hist.clear();  // plbfs_get_residual_history covers plbfs_run only
    fill_result(c, h, (float)ms, out);
    return h.status;
}

extern "C" int plbfs_get_residual_history(plbfs_ctx *c, double *out, int32_t max_steps) {
    if (!c || !out) return plbfs_fail(PLBFS_ERR_INPUT, "null argument");
    const size_t n = std::min((size_t)max_steps * 4, c->last_hist.size());
    std::memcpy(out, c->last_hist.data(), n * sizeof(double));
    return PLBFS_OK;
}

template <typename S>
static void launch_residual(plbfs_ctx *c, const DevMesh<S> &dm, double *Rd) {
    const V4<S> *st = (const V4<S> *)c->stA;
    V4<S> *grad = (V4<S> *)c->grad;
    hipLaunchKernelGGL(k_grad<S>, dim3(c->cell_grid), dim3(kBlock), 0, c->stream, dm, c->ctrl, st, grad);
    if (dm.n_border > 0)
        hipLaunchKernelGGL(k_flux_border<S>, dim3((dm.n_border + kBlock - 1) / kBlock), dim3(kBlock), 0, c->stream,
                           dm, c->prm, c->ctrl, st, grad);
    hipLaunchKernelGGL(k_residual_only<S>, dim3(c->L.n_blocks),
                       dim3(kBlock), c->lds_bytes, c->stream, dm, c->prm, st, grad, c->fbody, Rd);
}

extern "C" int plbfs_eval_residual(plbfs_ctx *c, double *grads, double *R) {
    if (!c) return plbfs_fail(PLBFS_ERR_INPUT, "null argument");
    if (int e = check_ghost_state(c)) return e;
    const int N = c->L.N;
    Ctrl h{};
    HIP_TRY(hipMemcpyAsync(c->ctrl, &h, sizeof(Ctrl), hipMemcpyHostToDevice, c->stream));
    double *Rd = c->stB;  // scratch: stB is rewritten before it is read in a step
    if (!c->f32) launch_residual<double>(c, c->dm, Rd);
    else launch_residual<float>(c, c->dm32, Rd);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(c->stream));
    if (grads) {
        // records of kGradRec V4 per cell, the gradient from V4 kGradOff on
        const int rs = 4 * (c->f32 ? kGradRec<float> : kGradRec<double>);
        const int ro = 4 * (c->f32 ? kGradOff<float> : kGradOff<double>);
        std::vector<double> h2((size_t)rs * N);
        if (!c->f32) {
            HIP_TRY(hipMemcpy(h2.data(), c->grad, h2.size() * sizeof(double), hipMemcpyDeviceToHost));
        } else {
            std::vector<float> h1((size_t)rs * N);
            HIP_TRY(hipMemcpy(h1.data(), c->grad, h1.size() * sizeof(float), hipMemcpyDeviceToHost));
            h2.assign(h1.begin(), h1.end());
        }
        for (int n = 0; n < N; n++)
            for (int q = 0; q < 12; q++) grads[(size_t)c->L.perm[n] * 12 + q] = h2[(size_t)rs * n + ro + q];
    }
    if (R) {
        std::vector<double> h4((size_t)4 * N);
        HIP_TRY(hipMemcpy(h4.data(), Rd, h4.size() * sizeof(double), hipMemcpyDeviceToHost));
        for (int n = 0; n < N; n++)
            for (int q = 0; q < 4; q++) R[(size_t)c->L.perm[n] * 4 + q] = h4[(size_t)q * N + n];
    }
    return PLBFS_OK;
}

extern "C" int plbfs_get_dt(plbfs_ctx *c, double *dt) {
    if (!c || !dt) return plbfs_fail(PLBFS_ERR_INPUT, "null argument");
    Ctrl h{};
    HIP_TRY(hipMemcpyAsync(c->ctrl, &h, sizeof(Ctrl), hipMemcpyHostToDevice, c->stream));
    int rc = launch_run_start(c, ctx_scratch(c));
    if (rc) return rc;
    HIP_TRY(hipStreamSynchronize(c->stream));
    double *outs[1] = {dt};
    return from_device_fields(c, c->dtl, 1, outs);
}

extern "C" int plbfs_enable_timing(plbfs_ctx *c, int32_t on) {
    if (!c) return plbfs_fail(PLBFS_ERR_INPUT, "null argument");
    c->timing = on != 0;
    for (auto &k : c->kstat) k = KStat();
    return PLBFS_OK;
}

extern "C" int plbfs_kernel_stats(plbfs_ctx *c, int32_t which, double *total_ms, int32_t *launches) {
    if (!c || which < 0 || which > 3) return plbfs_fail(PLBFS_ERR_INPUT, "bad arguments");
    if (total_ms) *total_ms = c->kstat[which].ms;
    if (launches) *launches = c->kstat[which].launches;
    return PLBFS_OK;
}

extern "C" int plbfs_layout_info(plbfs_ctx *c, int64_t *info) {
    if (!c || !info) return plbfs_fail(PLBFS_ERR_INPUT, "null argument");
    const Layout &L = c->L;
    int64_t slots = 0;
    for (int n = 0; n < L.N; n++) slots += L.st_cnt[n];
    info[0] = L.N;
    info[1] = L.F;
    info[2] = L.n_items;
    info[3] = slots;
    info[4] = L.G;
    info[5] = L.n_blocks;
    info[6] = L.max_items_per_block;
    info[7] = (int64_t)L.g_ent.size();
    info[8] = L.block_cells;
    info[9] = (int64_t)c->lds_bytes;
    return PLBFS_OK;
}

extern "C" int plbfs_get_body_force(plbfs_ctx *c, double *f) {
    if (!c || !f) return plbfs_fail(PLBFS_ERR_INPUT, "null argument");
    const int N = c->L.N;
    std::vector<double> h((size_t)3 * N);
    HIP_TRY(hipStreamSynchronize(c->stream));
    HIP_TRY(hipMemcpy(h.data(), c->fbody, h.size() * sizeof(double), hipMemcpyDeviceToHost));
    for (int n = 0; n < N; n++)
        for (int q = 0; q < 3; q++) f[(size_t)c->L.perm[n] * 3 + q] = h[(size_t)q * N + n];
    return PLBFS_OK;
}
