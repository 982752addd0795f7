// Per-cell and per-face pieces of one RK stage, shared by the single-case
// kernels (solver.hip) and the batched kernels (batch.hip).
//
// A "record index" names where cell c's state and gradient live: c for one
// case, c * B + b for case b of a batch stored case-fastest (so the B cases of
// one cell are adjacent and a gather of one cell for consecutive cases is one
// contiguous run).
#pragma once
#include <type_traits>

#include "lbfs_device.hpp"
#include "plbfs_hip.h"

namespace plbfs {

struct Rec1 {
    __device__ __forceinline__ size_t operator()(int c) const { return (size_t)c; }
};
struct RecB {
    unsigned B, b;  // unsigned: a product is one widening multiplication
    __device__ __forceinline__ size_t operator()(int c) const { return (size_t)(unsigned)c * B + b; }
    // first of cell c's three gradient V4, B apart ([cell][3][B])
    __device__ __forceinline__ size_t grad(int c) const { return (size_t)(unsigned)c * (3 * B) + b; }
};

// Per-cell RK accumulator between stages: the running sum t1 itself in FP64
// storage; in FP32 storage only the increment sum_k beta_k dt R_k (the
// conservative state stays in t0 in FP64, so small increments keep their bits).
template <typename S>
struct AccT {
    using type = double4;
};
template <>
struct AccT<float> {
    using type = float4;
};
template <typename S>
using Acc = typename AccT<S>::type;

struct StageArgs {
    double alpha, beta;
    int stage;  // 0..3
};

__device__ __forceinline__ double local_dt(const DevParams &prm, double visc, double rho, double u, double ax,
                                           double vol) {
    // Solver.cpp:1715-1744 with the x-slot-only CFL areas (A_y = A_z = 0)
    double eig = (fabs(u) + prm.ceff) * ax;
    eig = eig / prm.gamma;
    double ve = 2 * visc / prm.gamma / rho / vol;
    ve = ve * (ax * ax);
    eig = eig + 4 * ve;
    return prm.cfl * vol / eig;
}

template <typename T>
__device__ __forceinline__ T wave_sum(T x) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
    return x;
}

// Passes a value through an empty asm statement (no instruction is emitted).
// Without it the optimiser merges "load from LDS" and "load from global" on
// the two sides of a branch into one flat load through a selected pointer,
// which is slower than either and waits on both memory counters.
template <typename V>
__device__ __forceinline__ V opaque4(V v) {
    asm volatile("" : "+v"(v.x), "+v"(v.y), "+v"(v.z), "+v"(v.w));
    return v;
}

template <typename S, typename R>
struct GlobalStates {
    const V4<S> *__restrict__ st;
    R rec;
    __device__ __forceinline__ V4<S> operator()(int j) const { return st[rec(j)]; }
};

// States of cells [c0, c0 + nc) from an LDS copy, the rest from global memory.
template <typename S>
struct StagedStates {
    const V4<S> *__restrict__ st;
    const V4<S> *sSt;
    int c0, nc;
    __device__ __forceinline__ V4<S> operator()(int j) const {
        const unsigned rel = (unsigned)(j - c0);
        if (rel < (unsigned)nc) return opaque4(sSt[rel]);
        return st[j];
    }
};

// Least-squares gradient of cell i (src/gradients.cpp:319-389): folded stencil
// weights times neighbour differences; ghost neighbours from the owner's patch.
//
// The slots' indices are all loaded first, and the neighbours and weights of kSlots
// slots before their sums: with each slot's index behind the last slot's branch
// the loads are a chain of two latencies a slot (32^3 cavity in FP64 13.0 -> 11.2 us a
// launch, whatever the number of cells; 221k hexes in FP32 15.8 -> 13.1 us).  FP64
// takes one slot at a time: with two it holds 4 instead of 6 wavefronts per SIMD,
// and 384k tets take 23.0 instead of 20.3 us.
template <typename S, int kSlots, typename ST, typename W>
__device__ __forceinline__ void lsq_sums(const DevMesh<S> &m, int i, const int nbr[kMaxSlots], int cnt,
                                         const W &weight, const ST &state, S g[12]) {
    const auto none = [&](int s) { return kSlots == kMaxSlots && nbr[s] == kNoNbr; };
    const V4<S> q0 = state(i);
    const S p0[4] = {q0.x, q0.y, q0.z, q0.w};
#pragma unroll
    for (int q = 0; q < 12; q++) g[q] = (S)0;
#pragma unroll
    for (int s0 = 0; s0 < kMaxSlots; s0 += kSlots) {
        if (s0 >= m.max_slots) break;
        V4<S> qj[kSlots];
        S w[kSlots][3];
        int pb[kSlots];
#pragma unroll
        for (int u = 0; u < kSlots; u++) {
            const int s = s0 + u;
            if (s >= kMaxSlots || s >= m.max_slots) continue;
            // (periodic ghosts were replaced by their partner cell in st_nbr)
            qj[u] = state(nbr[s] >= 0 ? nbr[s] : i);
#pragma unroll
            for (int c = 0; c < 3; c++) w[u][c] = weight(s, c);
            if constexpr (kSlots == kMaxSlots) pb[u] = m.b_patch[nbr[s] < 0 && !none(s) ? -1 - nbr[s] : 0];
        }
#pragma unroll
        for (int u = 0; u < kSlots; u++) {
            const int s = s0 + u;
            if (s >= kMaxSlots || s >= m.max_slots) continue;
            S pj[4] = {qj[u].x, qj[u].y, qj[u].z, qj[u].w};
            if (nbr[s] < 0 && !none(s)) {
                const int b = -1 - nbr[s];
                const DevPatch P = m.patches[kSlots == kMaxSlots ? pb[u] : m.b_patch[b]];
                S fx[4] = {0, 0, 0, 0};
                if (P.flags & kGhostFixed) {
                    const V4<S> f = m.b_fix[b];
                    fx[0] = f.x; fx[1] = f.y; fx[2] = f.z; fx[3] = f.w;
                }
                ghost_state<S>(P, p0, p0, fx, pj);
            }
            if (s < cnt && !none(s)) {
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const S d = pj[q] - p0[q];
                    g[3 * q] += w[u][0] * d;
                    g[3 * q + 1] += w[u][1] * d;
                    g[3 * q + 2] += w[u][2] * d;
                }
            }
        }
    }
}

template <typename S, typename ST>
__device__ __forceinline__ void lsq_grad(const DevMesh<S> &m, int i, const ST &state, S g[12]) {
    int nbr[kMaxSlots];
#pragma unroll
    for (int s = 0; s < kMaxSlots; s++)
        if (s < m.max_slots) nbr[s] = m.st_nbr[(size_t)s * m.N + i];
    const auto weight = [&](int s, int c) { return m.st_w[((size_t)s * 3 + c) * m.N + i]; };
    lsq_sums<S, std::is_same<S, float>::value ? 3 : 1>(m, i, nbr, m.st_cnt[i], weight, state, g);
}

template <typename S>
__device__ __forceinline__ void unpack_side(V4<S> q, V4<S> a, V4<S> b, V4<S> d, S p[4], S g[12]) {
    p[0] = q.x;
    p[1] = q.y;
    p[2] = q.z;
    p[3] = q.w;
    g[0] = a.x; g[1] = a.y; g[2] = a.z; g[3] = a.w;
    g[4] = b.x; g[5] = b.y; g[6] = b.z; g[7] = b.w;
    g[8] = d.x; g[9] = d.y; g[10] = d.z; g[11] = d.w;
}

// Where a face item reads a cell's state and gradient: global memory, or with kStaged
// for cells of the block's own range [c0, c0 + nc) the copy the block staged in LDS
// (sRec: state, grad x3 per cell).  That choice is a branch a side, whose merge can
// wait for the owner's loads before the neighbour's are issued, so kernels that do not
// stage are built without it (flux of 4.1M tets in FP64 476 -> 439 us).  The batch keeps the gradients as [cell][3][B], so that
// consecutive cases of a cell are contiguous in each of the four loads.
template <typename S, typename R, bool kStaged>
struct SideLoader {
    const V4<S> *__restrict__ st;
    const V4<S> *__restrict__ grad;
    R rec;
    const V4<S> *sRec;  // staged records, cell-major then case lane: 4 * (rel * C + cl)
    int c0, nc;
    int C, cl;  // cases staged per cell and this item's case lane (1, 0 for one case)
    __device__ __forceinline__ void side(int c, S p[4], S g[12]) const {
        if constexpr (kStaged) {
            const unsigned rel = (unsigned)(c - c0);
            if (rel < (unsigned)nc) {
                const V4<S> *q = sRec + 4 * (rel * C + cl);
                unpack_side<S>(opaque4(q[0]), opaque4(q[1]), opaque4(q[2]), opaque4(q[3]), p, g);
                return;
            }
        }
        if constexpr (!std::is_same<R, Rec1>::value) {
            const V4<S> *gc = grad + rec.grad(c);
            unpack_side<S>(st[rec(c)], gc[0], gc[rec.B], gc[2 * rec.B], p, g);
        } else if constexpr (kGradOff<S> == 1) {
            const V4<S> *gc = grad + kGradRec<S> * (size_t)c;
            unpack_side<S>(gc[0], gc[1], gc[2], gc[3], p, g);
        } else {
            const V4<S> *gc = grad + kGradRec<S> * (size_t)c;
            unpack_side<S>(st[c], gc[0], gc[1], gc[2], p, g);
        }
    }
    __device__ __forceinline__ void sides(int o, int j, S po[4], S go[12], S pn[4], S gn[12]) const {
        side(o, po, go);
        side(j, pn, gn);
    }
};

// The same from LDS, where the block holds the records of every cell its items read:
// state and gradient, kLocalRec 16-byte pieces apart.  One piece more than a record
// has, so that the records of a wavefront's lanes start in all banks and not in two.
template <typename S>
constexpr int kLocalRec = sizeof(S) + 1;

template <typename S>
struct LocalLoader {
    const float4 *rec;
    uint32_t places;  // of the item's two cells (DevMesh::it_loc)
    static __device__ __forceinline__ void put(float4 *q, V4<S> st, const S g[12]) {
        S v[16] = {st.x, st.y, st.z, st.w};
#pragma unroll
        for (int k = 0; k < 12; k++) v[4 + k] = g[k];
#pragma unroll
        for (unsigned k = 0; k < sizeof(S); k++) __builtin_memcpy(q + k, reinterpret_cast<const char *>(v) + 16 * k, 16);
    }
    __device__ __forceinline__ void side(unsigned k, S p[4], S g[12]) const {
        const float4 *q = rec + kLocalRec<S> * k;
        S v[16];
#pragma unroll
        for (unsigned k = 0; k < sizeof(S); k++) __builtin_memcpy(reinterpret_cast<char *>(v) + 16 * k, q + k, 16);
#pragma unroll
        for (int k = 0; k < 4; k++) p[k] = v[k];
#pragma unroll
        for (int k = 0; k < 12; k++) g[k] = v[4 + k];
    }
    __device__ __forceinline__ void sides(int, int, S po[4], S go[12], S pn[4], S gn[12]) const {
        side(places & 0xffff, po, go);
        side(places >> 16, pn, gn);
    }
};

// Copies the records of cells [c0, c0 + nc) into LDS, 4 V4 per (cell, case
// lane) for the C cases b0 .. b0 + C - 1 of a batch of B (lanes past the last
// case are left unset); B = 0: a single case.
template <typename S>
__device__ __forceinline__ void stage_records(const V4<S> *__restrict__ st, const V4<S> *__restrict__ grad, int B,
                                              int b0, int C, int c0, int nc, V4<S> *sRec) {
    for (int k = threadIdx.x; k < nc * C * 4; k += blockDim.x) {
        const int r = k >> 2, q = k & 3;
        const int il = r / C, cl = r - il * C;
        if (B == 0) {
            if constexpr (kGradOff<S> == 1) sRec[k] = grad[kGradRec<S> * (size_t)(c0 + il) + q];
            else sRec[k] = q == 0 ? st[c0 + il] : grad[kGradRec<S> * (size_t)(c0 + il) + q - 1];
        } else if (b0 + cl < B) {
            const RecB rb{(unsigned)B, (unsigned)(b0 + cl)};
            sRec[k] = q == 0 ? st[rb(c0 + il)] : grad[rb.grad(c0 + il) + (size_t)(q - 1) * B];
        }
    }
}

// Byte offset of the staged records behind the face slots (C cases per slot)
// in a flux block's LDS.
template <typename S>
__host__ __device__ inline size_t staged_offset(int max_items, int C = 1) {
    return ((size_t)4 * max_items * C * sizeof(S) + 31) / 32 * 32;
}

// Dynamic LDS of one flux block: face slots, and with staging the block's own
// cell records for C cases.
template <typename S>
inline size_t flux_lds_bytes(int max_items, int block_cells, bool stage, int C = 1) {
    size_t b = staged_offset<S>(max_items, C);
    if (stage) b += (size_t)block_cells * C * 4 * sizeof(V4<S>);
    return b;
}

// Flux of face work item e (src/Solver.cpp:286-347 with populate_lattice_macros
// :840-1274); v3g = 3 nu / gamma of the case.  dtcap caps the item's streaming
// dt: a batch stores the geometric 0.5 sqrt(A) and caps it per case with
// 3 nu / (gamma fneq_min), the min the host applies for one case
// (src/unstructured_mesh.cpp:979-983); a single case passes infinity.
template <typename S>
struct Item {
    S geo[10];  // n A, owner offset, neighbour offset or n (each x, y, z), dt
    int2 on;
    unsigned side;
};

template <typename S>
__device__ __forceinline__ Item<S> load_item(const DevMesh<S> &m, unsigned e) {
    Item<S> it;
    S *geo = it.geo;
    const float4 *ip = m.it_p + ((size_t)(e >> 6) * (64 * kItemChunks<S>) + (e & 63));
    it.side = m.it_side[e];
    if constexpr (std::is_same<S, double>::value) {
        double2 q[kItemChunks<S>];
#pragma unroll
        for (int k = 0; k < kItemChunks<S>; k++) q[k] = __builtin_bit_cast(double2, ip[64 * k]);
        geo[0] = q[0].x; geo[1] = q[0].y; geo[2] = q[1].x; geo[3] = q[1].y; geo[4] = q[2].x;
        geo[5] = q[2].y; geo[6] = q[3].x; geo[7] = q[3].y; geo[8] = q[4].x;
        geo[9] = m.it_dt[e];
        it.on = __builtin_bit_cast(int2, q[4].y);
    } else {
        const float4 q0 = ip[0], q1 = ip[64], q2 = ip[128];
        geo[0] = q0.x; geo[1] = q0.y; geo[2] = q0.z; geo[3] = q0.w; geo[4] = q1.x;
        geo[5] = q1.y; geo[6] = q1.z; geo[7] = q1.w; geo[8] = q2.x; geo[9] = q2.y;
        it.on = int2{__float_as_int(q2.z), __float_as_int(q2.w)};
    }
    return it;
}

template <typename S, typename LD>
__device__ __forceinline__ void item_flux(const DevMesh<S> &m, const DevParams &prm, const Item<S> &it, const LD &ld,
                                          double v3g, double dtcap, S F[4]) {
    const S *geo = it.geo;
    const int o = it.on.x, nb = it.on.y;
    const S dt = fmin(geo[9], (S)dtcap);
    // the neighbour's record; for a boundary face that of its ghost's partner cell,
    // where it has one (and any record, not used, where it has none)
    int j = nb;
    if (nb < 0) {
        j = m.b_partner[-1 - nb];
        if (j < 0) j = o;
    }
    S po[4], go[12], pn[4], gN[12];
    ld.sides(o, j, po, go, pn, gN);
    // both sides' states at the face centre, as of an interior face.  FP32, whose batch
    // is bound by instructions, takes a chain of three (2% of a batch step); FP64 starts
    // with the gradients, which arrive before the states (4.1M tets 458 -> 439 us).
    S pI[4], pN[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        if constexpr (std::is_same<S, float>::value) {
            pI[q] = po[q] - geo[3] * go[3 * q] - geo[4] * go[3 * q + 1] - geo[5] * go[3 * q + 2];
            pN[q] = pn[q] - geo[6] * gN[3 * q] - geo[7] * gN[3 * q + 1] - geo[8] * gN[3 * q + 2];
        } else {
            pI[q] = po[q] - (geo[3] * go[3 * q] + geo[4] * go[3 * q + 1] + geo[5] * go[3 * q + 2]);
            pN[q] = pn[q] - (geo[6] * gN[3 * q] + geo[7] * gN[3 * q + 1] + geo[8] * gN[3 * q + 2]);
        }
    }
    if (nb < 0) {
        const int b = -1 - nb;
        const DevPatch P = m.patches[m.b_patch[b]];
        ghost_grad<S>(P, geo + 6, m.b_dmag[b], po, go, gN);
        if (b == 0) {
            // reconstructed like an interior face, from the ghost: the one whose index
            // equals n_cells (the reference's strict "neighbour > n_cells" test,
            // Solver.cpp:861)
            S pg[4], fx[4] = {0, 0, 0, 0};
            if (P.flags & kGhostFixed) {
                const V4<S> f = m.b_fix[0];
                fx[0] = f.x; fx[1] = f.y; fx[2] = f.z; fx[3] = f.w;
            }
            ghost_state<S>(P, po, pn, fx, pg);
#pragma unroll
            for (int q = 0; q < 4; q++)
                pN[q] = pg[q] - (m.b0[0] * gN[3 * q] + m.b0[1] * gN[3 * q + 1] + m.b0[2] * gN[3 * q + 2]);
        } else {
            if (P.rho_type == 1) pI[0] = (S)P.rho;
            else if (P.rho_type == 8) pI[0] = po[0];
            else pI[0] = po[0] - (geo[3] * gN[0] + geo[4] * gN[1] + geo[5] * gN[2]);
            if (P.vel_type == 1) {
                pI[1] = (S)P.u;
                pI[2] = (S)P.v;
                pI[3] = (S)P.w;
            } else if (P.vel_type == 8) {
                pI[1] = po[1];
                pI[2] = (S)0;
                pI[3] = po[3];
            } else {
#pragma unroll
                for (int q = 1; q < 4; q++)
                    pI[q] = po[q] - (geo[3] * gN[3 * q] + geo[4] * gN[3 * q + 1] + geo[5] * gN[3 * q + 2]);
            }
#pragma unroll
            for (int q = 0; q < 4; q++) pN[q] = pI[q];
        }
    }
    const S p0[4] = {(pI[0] + pN[0]) * (S)0.5, (pI[1] + pN[1]) * (S)0.5, (pI[2] + pN[2]) * (S)0.5,
                     (pI[3] + pN[3]) * (S)0.5};
    lattice_flux<std::is_same<S, float>::value, S>(geo, dt, (S)v3g, it.side, p0, pI, go, pN, gN, (S)prm.invgam,
                                                   (S)prm.c45, (S)prm.c15, (S)prm.rho0, F);
}

// Residual of cell i from its faces' LDS slots, summed in the reference's face
// order (src/Solver.cpp:353-366).  Slot sl of lane c lives at sF[q*stride + sl*C + c].
// The cell's entries are loaded together, from arrays that hold them face by face for
// all cells (2 B an entry).  Lists per cell behind an offset, 4 B an entry, are a
// dependent load and 16 B a tet more: 4.1M tets 488 -> 474 us in FP64, 288 -> 277 in
// FP32.
template <typename S>
struct CellFaces {
    int ent[kMaxSlots];  // without split borders
    double iv;
    float corr[3];  // FP32 with kAhead
};

template <typename S, bool kAhead = std::is_same<S, double>::value>
__device__ __forceinline__ CellFaces<S> load_faces(const DevMesh<S> &m, int i) {
    const size_t N = (size_t)m.N;
    CellFaces<S> in;
    in.iv = m.inv_vol[i];
    if (m.n_border == 0) {
#pragma unroll
        for (int s = 0; s < kMaxSlots; s++)
            if (s < m.max_ent) in.ent[s] = m.g_ent[s * N + i];
    }
    if constexpr (kAhead && std::is_same<S, float>::value) {
#pragma unroll
        for (int q = 0; q < 3; q++) in.corr[q] = m.corr[q * N + i];
    }
    return in;
}

// kAhead reads every slot before the first sum and holds them all: the flux kernel's FP32
// registers would spill (276 -> 400 us), so it is for FP64 and for k_stage.
template <typename S, bool kAhead = std::is_same<S, double>::value>
__device__ __forceinline__ void gather_residual(const DevMesh<S> &m, int i, const CellFaces<S> &in, const S *sF,
                                                int stride, int C, int c, double R[4], int B = 1, int b = 0) {
    const size_t N = (size_t)m.N;
    R[0] = R[1] = R[2] = R[3] = 0;
    // The signed fluxes are added (fma with +-1) and their sum divided by the volume: the
    // pressure fluxes through opposite faces, by far the largest terms, cancel exactly where
    // they are equal.  Divided one by one in the sum's fma they leave the first one's rounding,
    // the same way in every step: a box at rest moves, and the 32^3 cavity is 1.4 to 2.2e-13
    // from 64 bits after 200 steps instead of 0.7 to 1.1e-13.  Step in FP64 / FP32, that way and
    // this: 221k hexes 178.6 / 138.0 and 179.6 / 137.7 us, 32k 49.5 and 49.7, 59k 100.6 / 79.1 and
    // 100.8 / 78.7.
    auto add = [&](const S v[4], int own) {
        const double w = flip_sign(1.0, (unsigned)own, 0);
#pragma unroll
        for (int q = 0; q < 4; q++) R[q] = fma((double)v[q], w, R[q]);
    };
    auto slot = [&](int sl, S v[4]) {
#pragma unroll
        for (int q = 0; q < 4; q++) v[q] = sF[q * stride + (int)__umul24(sl, C) + c];
    };
    if (m.n_border == 0) {
        if constexpr (kAhead) {
            // (no face: slot 0, not added)
            S v[kMaxSlots][4];
#pragma unroll
            for (int s = 0; s < kMaxSlots; s++)
                if (s < m.max_ent) slot(in.ent[s] != kNoEnt ? in.ent[s] >> 1 : 0, v[s]);
#pragma unroll
            for (int s = 0; s < kMaxSlots; s++)
                if (s < m.max_ent && in.ent[s] != kNoEnt) add(v[s], in.ent[s] & 1);
        } else {
#pragma unroll
            for (int s = 0; s < kMaxSlots; s++) {
                if (s < m.max_ent && in.ent[s] != kNoEnt) {
                    S v[4];
                    slot(in.ent[s] >> 1, v);
                    add(v, in.ent[s] & 1);
                }
            }
        }
    } else {
        for (int s = 0; s < m.max_ent; s++) {
            const int ent = m.g_ent_split[s * N + i];
            if (ent < 0) break;
            S v[4];
            if (ent & 2) {
                // a face between two blocks: its flux was evaluated once by the border
                // pass, [4][n_border][B] with the case fastest (B = 1 for one case)
                const size_t j = (size_t)(ent >> 2), nbd = (size_t)m.n_border;
#pragma unroll
                for (int q = 0; q < 4; q++) v[q] = m.bflux[(q * nbd + j) * B + b];
            } else {
                slot(ent >> 2, v);
            }
            add(v, ent & 1);
        }
    }
    {
        // a product of its own, not fused with what a kernel adds to it
#pragma clang fp contract(off)
#pragma unroll
        for (int q = 0; q < 4; q++) R[q] = R[q] * in.iv;
    }
    if constexpr (std::is_same<S, float>::value) {
        // rho0/3 sum(+-n A)/V of the cell, omitted from the single-precision face fluxes
#pragma unroll
        for (int q = 0; q < 3; q++) R[1 + q] += (double)(kAhead ? in.corr[q] : m.corr[q * N + i]);
    }
}

// RK stage update of one cell record r (cell i) from its residual R
// (src/Solver.cpp:405-438, src/RungeKutta.h:16-18).  The last stage writes the
// new primitive solution, t0 and the next local time step, adds R^2 to sq and
// returns 1 for NaN or 2 for rho blow-up (src/Solver.cpp:448-493).
template <typename S>
struct RkIn {
    double dt;
    double4 t0;
    Acc<S> t1;             // behind the first stage
    double cfl_area, vol;  // last stage, with kAhead
};

template <typename S, bool kAhead = false>
__device__ __forceinline__ RkIn<S> load_rk(const DevMesh<S> &m, StageArgs sa, int i, size_t r, const double4 *t0,
                                           const Acc<S> *t1, const double *dtl) {
    RkIn<S> in;
    in.dt = dtl[r];
    in.t0 = t0[r];
    if (sa.stage != 0) in.t1 = t1[r];
    if (kAhead && sa.stage == 3) {
        in.cfl_area = m.cfl_area[i];
        in.vol = m.vol[i];
    }
    return in;
}

template <typename S, bool kAhead = false>
__device__ __forceinline__ int rk_update(const DevMesh<S> &m, const DevParams &prm, double visc, StageArgs sa,
                                         int i, size_t r, const RkIn<S> &in, const double R[4],
                                         V4<S> *__restrict__ st_out, double4 *__restrict__ t0,
                                         Acc<S> *__restrict__ t1, double *__restrict__ dtl, double sq[4],
                                         double &dt_next) {
    constexpr bool F32 = std::is_same<S, float>::value;
    const double dti = in.dt;
    const double4 ta = in.t0;
    const double a0 = ta.x, a1 = ta.y, a2 = ta.z, a3 = ta.w;
    // Solver.cpp:412-416
    double f1 = a0 + R[0] * dti * sa.alpha;
    double f2 = a1 + (R[1] + prm.force) * dti * sa.alpha;
    double f3 = a2 + R[2] * dti * sa.alpha;
    double f4 = a3 + R[3] * dti * sa.alpha;
    f2 = f2 / f1;
    f3 = f3 / f1;
    f4 = f4 / f1;
    // Solver.cpp:424-428
    const double db = dti * sa.beta;
    double b0, b1, b2, b3;
    if (!F32) {
        if (sa.stage == 0) {
            b0 = a0; b1 = a1; b2 = a2; b3 = a3;
        } else {
            const Acc<S> tb = in.t1;
            b0 = tb.x; b1 = tb.y; b2 = tb.z; b3 = tb.w;
        }
        b0 = b0 + db * R[0];
        b1 = b1 + db * (R[1] + prm.force);
        b2 = b2 + db * R[2];
        b3 = b3 + db * R[3];
    } else {
        // increments only; the conservative state is t0 + increments
        double d0 = 0, d1 = 0, d2 = 0, d3 = 0;
        if (sa.stage != 0) {
            const Acc<S> tb = in.t1;
            d0 = tb.x; d1 = tb.y; d2 = tb.z; d3 = tb.w;
        }
        d0 += db * R[0];
        d1 += db * (R[1] + prm.force);
        d2 += db * R[2];
        d3 += db * R[3];
        if (sa.stage < 3) {
            b0 = d0; b1 = d1; b2 = d2; b3 = d3;
        } else {
            b0 = a0 + d0; b1 = a1 + d1; b2 = a2 + d2; b3 = a3 + d3;
        }
    }
    const double r0 = F32 ? prm.rho0 : 0.0;  // single-precision density is stored as rho - rho0
    if (sa.stage < 3) {
        st_out[r] = V4<S>{(S)(f1 - r0), (S)f2, (S)f3, (S)f4};
        using E = typename std::conditional<F32, float, double>::type;
        t1[r] = Acc<S>{(E)b0, (E)b1, (E)b2, (E)b3};
        return 0;
    }
    // soln = t1 as primitives (Solver.cpp:431-436); it is the next step's temp
    const double s0 = b0, s1 = b1 / b0, s2 = b2 / b0, s3 = b3 / b0;
    st_out[r] = V4<S>{(S)(s0 - r0), (S)s1, (S)s2, (S)s3};
    t0[r] = double4{b0, b1, b2, b3};
    dt_next = prm.time_stepping == PLBFS_DT_CONSTANT
                  ? prm.cfl
                  : local_dt(prm, visc, s0, s1, kAhead ? in.cfl_area : m.cfl_area[i], kAhead ? in.vol : m.vol[i]);
    dtl[r] = dt_next;
    sq[0] += R[0] * R[0];
    sq[1] += R[1] * R[1];
    sq[2] += R[2] * R[2];
    sq[3] += R[3] * R[3];
    if (isnan(f1) || isnan(f2)) return 1;
    if (f1 / prm.ref_rho > 1000.0) return 2;
    return 0;
}

}  // namespace plbfs
