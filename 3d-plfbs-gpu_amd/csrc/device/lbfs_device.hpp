// Device-side data structures and numerics of the PLBFS solver (gfx950).
//
// Numerics follow the reference's CPU solver (src/Solver.cpp); the
// per-face equilibrium-flux evaluation is reorganised for registers:
// instead of materialising the 15 lattice populations (src/Solver.cpp:286-347,
// 655-837), each lattice point is reconstructed, its equilibrium evaluated and
// folded into running moments S0 = sum feq, S1 = sum e feq, Pi = sum e e^T feq.
// With f_k = feq_k(I) - tau (feq_k(I) - feq_k) and the D3Q15 isotropy
// sum w e_a e_b = I/3, sum w e_a e_b e_c e_d = (d_ab d_cd + d_ac d_bd + d_ad d_bc)/9,
// the reference's flux sums are exactly
//   sum_k e_k f_k       = (1 - tau) rho_I u_I + tau S1      (= S1, since rho_I u_I = S1)
//   sum_k e_k e_k^T f_k = (1 - tau) rho_I (I/3 + u_I u_I^T / gamma) + tau Pi
// so only S0, S1 and Pi are needed, summed from the pairs of opposite points and
// weighted once per face.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace plbfs {

// flags: the ghost gradient copies cell b_partner[b]'s (periodic partner, or
// cell 0 where the reference's update leaves the ghost unwritten), and the
// ghost state holds per-ghost fixed values b_fix[b] (those patches)
constexpr int32_t kGhostGradFromCell = 1;
constexpr int32_t kGhostFixed = 2;

struct DevPatch {
    int32_t rho_type, vel_type, is_empty, flags;
    double rho, u, v, w;
};

// Step control block, written by the reduction kernel, read by every kernel.
struct Ctrl {
    int32_t done;    // nonzero: skip all further work
    int32_t status;  // 0 ok, PLBFS_ERR_NAN, PLBFS_ERR_RHO, PLBFS_ERR_IBM
    int32_t step;    // steps completed in this run
    int32_t converged;
    int32_t rebuild;  // nonzero: an immersed node drifted half its list margin
    unsigned long long arrived;  // blocks of the step's last kernel so far; 0 between kernels
    double res[4];
};

// Per-cell records gathered by neighbours are stored array-of-structures so a
// gather touches one 32 B (state) or 96 B (gradient) run instead of 4 or 12
// separate cache lines.
template <typename S>
struct V4T;
template <>
struct V4T<double> {
    using type = double4;
};
template <>
struct V4T<float> {
    using type = float4;
};
template <typename S>
using V4 = typename V4T<S>::type;

// Gradient records gathered by the face items of a single case.  FP64: three V4
// (d/dx, d/dy, d/dz of rho, u, v, w), 96 B.  FP32: the cell's state followed by its
// three gradient V4, 64 B, so that a face side is one aligned 64 B run; the
// gradient kernel writes all four (the state it read).
template <typename S>
inline constexpr int kGradRec = std::is_same<S, float>::value ? 4 : 3;  // V4 per record
template <typename S>
inline constexpr int kGradOff = std::is_same<S, float>::value ? 1 : 0;  // first gradient V4

// Workgroups are dispatched round-robin over the 8 XCDs (blockIdx.x mod 8), and
// each XCD has its own L2.  Remapping gives XCD x a contiguous range of logical
// blocks, so Hilbert-adjacent cells (and their shared halo) meet in one L2.
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_block(int bid, int nblk, int remap) {
    if (!remap) return bid;
    const int q = nblk / kXcds, r = nblk % kXcds;
    const int x = bid % kXcds, k = bid / kXcds;
    return x * q + (x < r ? x : r) + k;
}

constexpr int kNoEnt = 0xffff;  // no face (see DevMesh::g_ent)

// 16 B chunks per face item (see DevMesh::it_p).
template <typename S>
inline constexpr int kItemChunks = std::is_same<S, float>::value ? 3 : 5;

template <typename S>
struct DevMesh {
    int N, G, n_blocks, max_items;
    // border items [border0, border0 + n_border) and their fluxes [4][n_border]
    // (one evaluation per face between two blocks; 0 when items are duplicated)
    int64_t border0;
    int n_border;
    S *bflux;
    int xcd_remap;
    int block_cells;  // cells per flux block (a multiple of 8)
    int stage;        // 1: flux blocks stage their own cells' records in LDS
    int grad_stage;   // 1: gradient blocks stage their own cells' states in LDS
    int max_slots;    // most stencil slots of a cell
    int64_t E;
    const uint8_t *st_cnt;
    const int32_t *st_nbr;
    const S *st_w;
    const double *vol, *inv_vol, *cfl_area;
    const int32_t *blk_item_off;
    // Face work items in groups of 64: chunk k of item e, 16 B, is it_p[((e >> 6)
    // * kItemChunks<S> + k) * 64 + (e & 63)], so that every load of a wavefront of
    // consecutive items is one contiguous KiB (16 B a lane at a record's stride
    // takes the address unit two to three times as long).  An item is the area
    // vector n A, the owner's centroid and the neighbour's centroid from the face
    // centre, each (x, y, z); the streaming dt (FP32 here, FP64 in it_dt); and the
    // owner and neighbour (or -1-b) as two ints.  A boundary face holds its unit
    // normal in the neighbour's place: its ghost's centroid is only used on boundary
    // face 0, as b0.  it_side holds the lattice side bits (see side_point).
    const float4 *it_p;
    const double *it_dt;
    const uint16_t *it_side;
    // k_stage: the cells that a flux block's items read, max_local places a block, their
    // stencil neighbours (slot by slot; kNoNbr behind the last) and weights (st_w, slot
    // after slot in pieces of 16 B, piece k of place p at k * n_places + p) and an item's
    // two places
    const int32_t *loc_cell, *loc_nbr;
    const float4 *loc_w;
    const uint32_t *it_loc;
    int max_local, n_places, n_patches;
    S b0[3];
    // a cell's faces in the reference face order, entry s of cell i at s * N + i:
    // slot << 1 | is_owner, kNoEnt behind the last one (max_ent: most of a cell);
    // with a border pass g_ent_split instead, as in the layout, -1 behind the last
    const uint16_t *g_ent;
    const int32_t *g_ent_split;
    int max_ent;
    // [n_blocks] nonzero where a flux block holds a cell the immersed boundary
    // spreads force to; null: every block reads the body force
    const int32_t *blk_force;
    const int32_t *b_patch;
    const int32_t *b_partner;  // cell whose gradient the ghost takes (kGhostGradFromCell), -1 elsewhere
    const V4<S> *b_fix;        // [G] fixed ghost states (kGhostFixed); FP32: rho - rho0
    const S *b_dmag;
    const DevPatch *patches;  // FP32 storage: rho values shifted by -rho0
    const S *corr;            // FP32 storage: [3][N] rho0/3 sum(+-n A)/V per cell
};

struct DevParams {
    double visc, gamma, invgam, visc3_invgam, c45, c15, force, cfl, ceff, ref_rho, ref_mom, tol;
    double rho0;  // FP32 storage: density offset (rho = rho0 + stored value)
    int time_stepping;
    int use_body_force;
};

// ---------------------------------------------------------------------------
// Ghost cells (src/Solution.cpp:759-833, src/gradients.cpp:395-504,592-648)
// ---------------------------------------------------------------------------

// pp: state of the periodic partner (read only by type 3); fx: the ghost's
// fixed values (read only by the types the reference's update leaves at the
// ghost's initial state, and the parabolic u, v of types 4 and 5).
template <typename T>
__device__ __forceinline__ void ghost_state(const DevPatch &P, const T po[4], const T pp[4], const T fx[4],
                                            T pg[4]) {
    // selects between values at hand: a chain of branches costs each slot of a small
    // mesh's wavefronts the latency of every branch's loads
    const int rt = P.rho_type, vt = P.vel_type;
    const T b[4] = {(T)P.rho, (T)P.u, (T)P.v, (T)P.w};
    const bool rfix = rt == 4 || rt == 5 || rt == 9, vfix = vt == 4 || vt == 5 || vt == 7 || vt == 9;
    T r = po[0];  // 2 (neumann, dx = 0) and 8 (symmetry)
    r = rt == 3 ? pp[0] : r;
    r = rfix ? fx[0] : r;
    r = rt == 6 || rt == 7 ? b[0] : r;
    r = rt == 1 ? b[0] - (po[0] - b[0]) : r;
    pg[0] = r;
#pragma unroll
    for (int q = 1; q < 4; q++) {
        T v = po[q];
        if (q == 2) v = vt == 8 ? -po[q] : v;
        v = vt == 3 ? pp[q] : v;
        v = vfix ? fx[q] : v;
        v = vt == 6 ? b[q] : v;
        v = vt == 1 ? b[q] - (po[q] - b[q]) : v;
        pg[q] = v;
    }
}

// Ghost gradient gg from the owner's state and gradient.  On entry gg is the
// gradient of cell b_partner[b], which type 3 and the types whose ghost the
// reference's update leaves unwritten keep (other patches have no partner; what gg
// holds is not used).  rho_type 8 leaves the reference's zero-initialised rho
// slot untouched, so it is zero here too.
template <typename T>
__device__ __forceinline__ void ghost_grad(const DevPatch &P, const T n[3], T dmag, const T po[4], const T go[12],
                                           T gg[12]) {
    const int rt = P.rho_type, vt = P.vel_type;
    if (rt == 1) {
        const T q = (T)2 * ((T)P.rho - po[0]) / dmag;
        gg[0] = q * n[0];
        gg[1] = q * n[1];
        gg[2] = q * n[2];
    } else if (rt == 2) {
        gg[0] = go[0] * ((T)1 - n[0]);
        gg[1] = go[1] * ((T)1 - n[1]);
        gg[2] = go[2] * ((T)1 - n[2]);
    } else if (rt == 7) {
        gg[0] = go[0];
        gg[1] = go[1];
        gg[2] = go[2];
    } else if (!(rt == 3 || rt == 4 || rt == 5 || rt == 9)) {
        gg[0] = gg[1] = gg[2] = (T)0;
    }
    if (vt == 1 || vt == 8) {
        const T qu = (T)2 * ((T)P.u - po[1]) / dmag;
        const T qv = (T)2 * ((T)P.v - po[2]) / dmag;
        const T qw = (T)2 * ((T)P.w - po[3]) / dmag;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            gg[3 + c] = qu * n[c];
            gg[6 + c] = qv * n[c];
            gg[9 + c] = qw * n[c];
        }
    } else if (vt == 2) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
            gg[3 + c] = go[3 + c] * ((T)1 - n[c]);
            gg[6 + c] = go[6 + c] * ((T)1 - n[c]);
            gg[9 + c] = go[9 + c] * ((T)1 - n[c]);
        }
    } else if (!(vt == 3 || vt == 4 || vt == 5 || vt == 7 || vt == 9)) {
#pragma unroll
        for (int q = 3; q < 12; q++) gg[q] = (T)0;
    }
}

// ---------------------------------------------------------------------------
// Lattice evaluation (src/Solver.cpp:840-1374 restructured as moments)
// ---------------------------------------------------------------------------

// e.g of one lattice direction from a gradient triple g (x, y, z) and its sum
// s = gx + gy + gz: the four body diagonals share s.
template <int EX, int EY, int EZ, typename T>
__device__ __forceinline__ T dir_deriv(const T *g, T s) {
    if constexpr (EX != 0 && EY != 0 && EZ != 0) {
        // EX, EY, EZ in {+-1}: at most one of them is -1 in the pairs' order
        if constexpr (EX < 0) return s - (T)2 * g[0];
        else if constexpr (EY < 0) return s - (T)2 * g[1];
        else if constexpr (EZ < 0) return s - (T)2 * g[2];
        else return s;
    } else {
        // (no products with zero: the compiler may not drop them, 0 x inf is NaN)
        return g[EX ? 0 : (EY ? 1 : 2)];
    }
}

// e.u of a lattice direction (axis directions are +1 here).
template <int EX, int EY, int EZ, typename T>
__device__ __forceinline__ T dir_dot(T u, T v, T w) {
    if constexpr (EX == 0 && EY == 0 && EZ == 0) return (T)0;
    else if constexpr (EX != 0 && EY != 0 && EZ != 0) return (T)EX * u + (T)EY * v + (T)EZ * w;
    else return EX ? u : (EY ? v : w);
}

// Equilibrium at state (r, u, v, w) divided by the lattice weight, for the
// direction +-e with s3 = +-3.  With DEV (FP32 storage) the density is a deviation
// r = rho - rho0 and the value returned is h = (feq - w rho0) / w =
// r (1 + X) + rho0 X, X = 3 e.u + (4.5 (e.u)^2 - 1.5 u^2)/gamma, so the O(1) part
// rho0 never enters single precision.
template <int EX, int EY, int EZ, bool DEV, typename T>
__device__ __forceinline__ T pop_eq(T r, T u, T v, T w, T s3, T c45, T c15, T rho0) {
    const T eu = dir_dot<EX, EY, EZ, T>(u, v, w);
    const T usq = u * u + v * v + w * w;
    // X = +-3 e.u + (4.5 (e.u)^2 - 1.5 u^2) / gamma, as e.u (s3 + c45 e.u) - c15 u^2
    // with c45 = 4.5 / gamma and c15 = 1.5 / gamma
    const bool rest = EX == 0 && EY == 0 && EZ == 0;
    const T X = rest ? -(c15 * usq) : eu * (s3 + c45 * eu) - c15 * usq;
    if constexpr (DEV) return r + (r + rho0) * X;
    else return r + r * X;
}

// Passes a value through an empty asm statement (no instruction is emitted), so
// that what follows is not merged with another use of the same value.
template <typename T>
__device__ __forceinline__ T opaque(T x) {
    asm volatile("" : "+v"(x));
    return x;
}

// x with its sign flipped where bit k of `bits` is set.
template <typename T>
__device__ __forceinline__ T flip_sign(T x, unsigned bits, int k) {
    const unsigned m = (bits << (31 - k)) & 0x80000000u;
    if constexpr (std::is_same<T, float>::value) return __uint_as_float(__float_as_uint(x) ^ m);
    else return __hiloint2double(__double2hiint(x) ^ (int)m, __double2loint(x));
}

// Lattice pairs +e / -e (pair index P: x, y, z, then the four body diagonals).
// Point +e takes the neighbour side iff e.n < 0 and point -e iff e.n > 0 (the
// reference's "sum of signed normal components > 0" tests,
// src/Solver.cpp:958-1273).  So with d = e or -e, whichever points from the owner
// to the neighbour, +d always comes from the owner side and -d from the neighbour
// side, except where e.n = 0: there both come from the owner side.  The host
// decides both in FP64: bit P of `side` is set where d = -e (e.n < 0), bit 7 + P
// where e.n = 0.  (For faces containing a lattice direction e.n is zero
// analytically and its sign is rounding noise, so evaluating it in another
// precision would pick the other side.)
//
// One side's seven points, h[P] at +d (OUT) or -d of every pair: p is the side's
// state at the face centre, g its gradient.
constexpr int kPairs = 7;

//
// The owner side's pass replaces hb[P], the neighbour side's value at -d, by its own
// where e.n = 0; a wavefront without such a face skips that by a scalar branch.
template <int P, int EX, int EY, int EZ, bool OUT, bool DEV, typename T>
__device__ __forceinline__ void side_point(unsigned side, T dt, const T p[4], const T g[12], const T s[4], T c45,
                                           T c15, T rho0, T *h, T *hb) {
    // the point that streams along +-d starts at -(+-d) dt from the face centre; +-d is e times a sign
    const T tau = opaque(flip_sign<T>(OUT ? -dt : dt, side, P));
    const T s3 = flip_sign<T>(OUT ? (T)3 : (T)-3, side, P);
    T d[4];
#pragma unroll
    for (int q = 0; q < 4; q++) d[q] = dir_deriv<EX, EY, EZ, T>(g + 3 * q, s[q]);
    // one point after the other (tau and h are passed through opaque in this
    // order): interleaved for instruction-level parallelism, which other wavefronts
    // provide already, the points would take some 40 registers more
    h[P] = opaque(pop_eq<EX, EY, EZ, DEV, T>(p[0] + tau * d[0], p[1] + tau * d[1], p[2] + tau * d[2],
                                             p[3] + tau * d[3], s3, c45, c15, rho0));
    if constexpr (OUT) {
        const bool both = (side & (1u << (kPairs + P))) != 0;
        if (__builtin_amdgcn_ballot_w64(both) != 0) {
            const T ho = pop_eq<EX, EY, EZ, DEV, T>(p[0] - tau * d[0], p[1] - tau * d[1], p[2] - tau * d[2],
                                                    p[3] - tau * d[3], -s3, c45, c15, rho0);
            hb[P] = both ? ho : hb[P];
        }
    }
}

template <bool OUT, bool DEV, typename T>
__device__ __forceinline__ void side_points(unsigned side, T dt, const T p[4], const T g[12], T c45, T c15, T rho0,
                                            T h[kPairs], T hb[kPairs]) {
    T s[4];
#pragma unroll
    for (int q = 0; q < 4; q++) s[q] = g[3 * q] + g[3 * q + 1] + g[3 * q + 2];
    side_point<0, 1, 0, 0, OUT, DEV, T>(side, dt, p, g, s, c45, c15, rho0, h, hb);
    side_point<1, 0, 1, 0, OUT, DEV, T>(side, dt, p, g, s, c45, c15, rho0, h, hb);
    side_point<2, 0, 0, 1, OUT, DEV, T>(side, dt, p, g, s, c45, c15, rho0, h, hb);
    side_point<3, 1, 1, 1, OUT, DEV, T>(side, dt, p, g, s, c45, c15, rho0, h, hb);
    side_point<4, 1, 1, -1, OUT, DEV, T>(side, dt, p, g, s, c45, c15, rho0, h, hb);
    side_point<5, 1, -1, 1, OUT, DEV, T>(side, dt, p, g, s, c45, c15, rho0, h, hb);
    side_point<6, -1, 1, 1, OUT, DEV, T>(side, dt, p, g, s, c45, c15, rho0, h, hb);
}

// Reciprocal: correctly rounded in FP64; in FP32 the hardware estimate
// (1 ulp), whose error is far below the FP32 variant's tolerance.
template <typename T>
__device__ __forceinline__ T lattice_rcp(T x) {
    if constexpr (std::is_same<T, float>::value) return __builtin_amdgcn_rcpf(x);
    else return (T)1 / x;
}

// Flux through a face with area vector nA (owner -> neighbour); tau is passed as
// its parts v3g / dt.  With DEV the momentum flux omits the constant rho0/3 n A, whose sum over a cell's faces is a per-cell geometric
// constant added separately.
//
// The two sides are evaluated one after the other, seven points each, so only one
// side's gradient is live with the other side's seven values.  Evaluating only
// the side each point comes from (instead of both, and a select) halves the
// reconstruction.  The second evaluation that e.n = 0 needs is skipped by a
// wavefront without such a face (all interior faces of a jittered mesh).
template <bool DEV, typename T>
__device__ __forceinline__ void lattice_flux(const T nA[3], T dt, T v3g, unsigned side, const T p0[4],
                                             const T pI[4], const T gO[12], const T pN[4], const T gN[12], T invgam,
                                             T c45, T c15, T rho0, T F[4]) {
    const T w0 = (T)(2.0 / 9.0), w1 = (T)(1.0 / 9.0), w7 = (T)(1.0 / 72.0);
    const T h0 = pop_eq<0, 0, 0, DEV, T>(p0[0], p0[1], p0[2], p0[3], (T)3, c45, c15, rho0);
    __builtin_amdgcn_sched_barrier(0);
    T ha[kPairs], hb[kPairs];
    side_points<false, DEV, T>(side, dt, pN, gN, c45, c15, rho0, hb, hb);
    side_points<true, DEV, T>(side, dt, pI, gO, c45, c15, rho0, ha, hb);
    // pair sums S = h(+e) + h(-e) (even moments) and differences D = h(+e) - h(-e)
    T S[kPairs], D[kPairs];
#pragma unroll
    for (int k = 0; k < kPairs; k++) {
        S[k] = ha[k] + hb[k];
        D[k] = flip_sign<T>(ha[k] - hb[k], side, k);
    }
    // weighted moments: S0, S1 and Pi; each axis pair feeds one component of
    // every moment, the four diagonals all of them
    const T a = S[3] + S[4], b = S[5] + S[6], c = S[3] - S[4], d = S[5] - S[6];
    const T e = D[3] + D[4], f = D[5] - D[6];
    const T dS = w7 * (a + b);
    const T s0 = w0 * h0 + w1 * (S[0] + S[1] + S[2]) + dS;
    const T sx = w1 * D[0] + w7 * (e + f);
    const T sy = w1 * D[1] + w7 * (e - f);
    const T sz = w1 * D[2] + w7 * ((D[3] - D[4]) + (D[5] + D[6]));
    const T pxx = w1 * S[0] + dS, pyy = w1 * S[1] + dS, pzz = w1 * S[2] + dS;
    const T pxy = w7 * (a - b), pxz = w7 * (c + d), pyz = w7 * (c - d);
    const T tau = v3g * lattice_rcp(dt);
    const T rI = DEV ? rho0 + s0 : s0;
    const T ir = lattice_rcp(rI);
    const T ux = sx * ir, uy = sy * ir, uz = sz * ir;
    const T om = (T)1 - tau;
    // sum e e^T feq(I) = rho_I (I/3 + u u^T/gamma); in DEV form rho0 I/3 is dropped
    const T iso = DEV ? s0 * (T)(1.0 / 3.0) : rI * (T)(1.0 / 3.0);
    const T k = om * rI * invgam, m0 = om * iso;
    const T kx = k * ux, ky = k * uy, kz = k * uz;
    const T mxx = m0 + tau * pxx + kx * ux;
    const T myy = m0 + tau * pyy + ky * uy;
    const T mzz = m0 + tau * pzz + kz * uz;
    const T mxy = tau * pxy + kx * uy;
    const T mxz = tau * pxz + kx * uz;
    const T myz = tau * pyz + ky * uz;
    F[0] = sx * nA[0] + sy * nA[1] + sz * nA[2];
    F[1] = mxx * nA[0] + mxy * nA[1] + mxz * nA[2];
    F[2] = mxy * nA[0] + myy * nA[1] + myz * nA[2];
    F[3] = mxz * nA[0] + myz * nA[1] + mzz * nA[2];
}

}  // namespace plbfs
