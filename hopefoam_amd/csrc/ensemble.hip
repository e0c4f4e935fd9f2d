// Ensembles of independent LDG advection-diffusion cases (u_t + div(a u) = nu div(q), q = grad u; periodic
// triangle meshes of different sizes and orders) for gfx950.  The method is the local discontinuous
// Galerkin scheme of Cockburn & Shu (1998) with alternating fluxes (u^ from the side the switch vector
// points away from, q^ from the other, penalty tau on u jumps) in the nodal strong form; it has no
// counterpart in the reference, whose dgc::laplacian is empty.
//
// Each LSERK4 stage is two passes (the auxiliary q of an element's neighbours must be complete before the
// right-hand side reads it -- a grid-wide dependency that a kernel boundary settles without fences or spin
// waits), each pass one persistent launch per order present in the ensemble over all cases of that order:
//   ens_kernel<0, N, P>  q = grad u - LIFT(fscale n (u- - u^))                   -> qx, qy
//   ens_kernel<1, N, P>  rhs = -div(a u - nu q) + LIFT(fscale (n.F- - n.F^)), then res = a res + dt rhs,
//                        u_next = u + b res
// Orders (and row splits) get kernels of their own so that each is register-allocated for its own shape
// (one kernel holding every order needs the union of all their registers, and spills).
// A work item is a run of 64-element blocks of one case, taken by a whole workgroup of kEnsWaves waves: one
// element per lane, each block's node rows split into P slices, the (block, slice) tasks spread over the waves.
// All lanes of a wave need the same operator entry at a time, so the order's operators (transposed, rows
// padded to kEnsRows with zeros: the R entries of one column a slice needs are contiguous and need no
// clamping) sit in LDS and are read as broadcasts.  Element and face loads are issued in batches ahead of
// the arithmetic that consumes them.
// The slice count P per order (rows per lane R = ceil(Np / P) <= 8) is the tile shape the autotuner picks.
// Each order's items are split into 8 contiguous ranges of equal estimated cost, one per XCD, so that the
// neighbour traces an item reads were brought into the same XCD's L2 by the items next to it.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "ensemble.hpp"
#include "lds_stage.hpp"

namespace dg {

__host__ __device__ constexpr int ens_np(int N) { return (N + 1) * (N + 2) / 2; }
__host__ __device__ constexpr int ens_rows(int N, int P) { return (ens_np(N) + P - 1) / P; }
__host__ __device__ constexpr bool ens_split_ok(int N, int P) {
    return N >= 1 && N <= 8 && (P == 1 || P == 2 || P == 4 || P == 8) && ens_rows(N, P) <= 8 &&
           (P == 1 || ens_rows(N, P) >= 2);
}

bool ens_split_supported(int N, int P) { return P == kEnsMfma ? (N >= 2 && N <= 8) : ens_split_ok(N, P); }

// node of point k of face f (face f runs from vertex f to vertex f + 1; row j of the nodal set holds
// N + 1 - j nodes and starts at j (N + 1) - j (j - 1) / 2)
template <int N>
__device__ __forceinline__ int face_node(int f, int k) {
    if (f == 0) return k;
    if (f == 1) return k * (N + 1) - k * (k - 1) / 2 + (N - k);
    const int j = N - k;
    return j * (N + 1) - j * (j - 1) / 2;
}

__device__ __forceinline__ size_t nidx(int e, int n, int Np) { return (size_t(e >> 4) * Np + n) * 16 + (e & 15); }

using d4_t = double __attribute__((ext_vector_type(4)));
__device__ __forceinline__ d4_t mfma64(double a, double b, d4_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// MFMA variant: a wave owns 16 elements (group grp of the case); lane (col, rg) = (lane % 16, lane / 16).
// B operands: K step s of the volume products holds node 4 s + rg of element col; K step k of the lift holds point k
// of face rg (the fragments' fourth row of a step is zero), so a lane reads the geometry, the neighbour and its
// address of one face only.  A operands: the operator fragments in LDS.
// Accumulators: register r of row tile m holds row 16 m + rg + 4 r of element col, node 4 s + rg with s = 4 m + r:
// a lane owns the same nodes on both sides of the products, and the update has u in registers.
// The passes are bound by latency (an ensemble's order rarely has more than two groups per SIMD), so everything a
// group needs is requested before anything is used: one memory latency for the group's own values and connectivity,
// one for the neighbours'.  Microseconds per stage (both passes) of 7 to 13 cases of one order, elements in all, with a
// face's points running over the K steps, face geometry per point and the loads left where the products need them -> now:
//   order 8, 50048: 82 -> 60    6, 36136: 41.6 -> 35.5    5, 30076: 30.4 -> 28.9    4, 16404: 15.2 -> 12.7
//   order 7, 20634: 32.4 -> 27.5 (the lift takes eight matrix steps in place of six)   3, 20918: 12.2 -> 11.1
template <int N>
struct EnsLane {
    const double *up;       // u of the neighbour's node 0
    unsigned own[N + 1];    // offset of point k of the lane's face in the group's nodes
    unsigned nbr[N + 1];    // the matching point's offset from up
    double nx, ny, fs, tf;
    bool own_side;
};

// offset (in values, 16 per node) of point k of face f, f varying over the lanes
template <int N>
__device__ __forceinline__ unsigned face_off(int f, int k) {
    return 16u * unsigned(f == 0 ? face_node<N>(0, k) : f == 1 ? face_node<N>(1, k) : face_node<N>(2, k));
}

// the lane's face (face 2 on the fourth row) of its element; ug: u of the group, ue: u of element 0
template <int N>
__device__ __forceinline__ void ens_lane(const EnsArgs& a, const EnsCase& cs, const double* u, int grp, int col, int rg,
                                         EnsLane<N>& L) {
    constexpr int Np = ens_np(N);
    const unsigned Kp = cs.Kp, e = unsigned(grp) * 16 + col, f = rg < 3 ? rg : 2;
    const double* g = a.geo + cs.off_geo;
    const int c = (a.conn + cs.off_conn)[f * Kp + e];
    L.nx = g[(4 + 4 * f) * Kp + e];
    L.ny = g[(5 + 4 * f) * Kp + e];
    L.fs = g[(6 + 4 * f) * Kp + e];
    L.tf = g[(7 + 4 * f) * Kp + e];
    const int en = c >> 3, fn = (c >> 1) & 3;
    L.own_side = c & 1;
    L.up = u + size_t(en >> 4) * (Np * 16) + (en & 15);
#pragma unroll
    for (int k = 0; k <= N; ++k) {
        L.own[k] = face_off<N>(f, k) + col;
        L.nbr[k] = face_off<N>(fn, N - k);
    }
}

// One group's inputs of the q pass, requested together
template <int N>
struct EnsQIn {
    double ub[ens_mfma_ks(N)], um[N + 1], up[N + 1], m[4];
    double nx, ny, fs;
    bool own_side;
};

template <int N>
__device__ __forceinline__ void ens_q_load(const EnsArgs& a, const EnsCase& cs, int grp, int lane, EnsQIn<N>& in) {
    constexpr int Np = ens_np(N), KS = ens_mfma_ks(N);
    const int left = cs.K - grp * 16, c0 = lane & 15, col = c0 < left ? c0 : left - 1, rg = lane >> 4;
    const size_t arr = size_t(cs.Kp) * Np;
    const double* u = a.data + cs.off_u + size_t(a.cur) * arr;
    const double* ug = u + size_t(grp) * (Np * 16);
    const double* g = a.geo + cs.off_geo + grp * 16;
    EnsLane<N> L;
    ens_lane<N>(a, cs, u, grp, col, rg, L);
#pragma unroll
    for (int s = 0; s < KS; ++s) in.ub[s] = 4 * s + rg < Np ? ug[unsigned(64 * s + 16 * rg + col)] : 0.0;
#pragma unroll
    for (int k = 0; k <= N; ++k) in.um[k] = ug[L.own[k]];
#pragma unroll
    for (int i = 0; i < 4; ++i) in.m[i] = (g + size_t(i) * cs.Kp)[unsigned(col)];
#pragma unroll
    for (int k = 0; k <= N; ++k) in.up[k] = L.up[L.nbr[k]];
    in.nx = L.nx;
    in.ny = L.ny;
    in.fs = L.fs;
    in.own_side = L.own_side;
}

template <int N>
__device__ __forceinline__ void ens_q_mfma(const EnsArgs& a, const EnsCase& cs, const double* ops, int grp, int lane,
                                           const EnsQIn<N>& in) {
    constexpr int Np = ens_np(N), Nfp = N + 1;
    constexpr int MT = ens_mfma_mt(N), KS = ens_mfma_ks(N);
    const int rg = lane >> 4;
    const size_t arr = size_t(cs.Kp) * Np;
    const double* DrF = ops;
    const double* DsF = ops + MT * KS * 64;
    const double* LF = ops + 2 * MT * KS * 64;
    d4_t ar[MT], as[MT], lx[MT], ly[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) ar[m] = as[m] = lx[m] = ly[m] = d4_t{0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            ar[m] = mfma64(DrF[(m * KS + s) * 64 + lane], in.ub[s], ar[m]);
            as[m] = mfma64(DsF[(m * KS + s) * 64 + lane], in.ub[s], as[m]);
        }
#pragma unroll
    for (int k = 0; k < Nfp; ++k) {
        const double d = in.own_side ? 0.0 : in.fs * (in.um[k] - in.up[k]);
        const double gx = in.nx * d, gy = in.ny * d;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const double L = LF[(m * Nfp + k) * 64 + lane];
            lx[m] = mfma64(L, gx, lx[m]);
            ly[m] = mfma64(L, gy, ly[m]);
        }
    }
    const bool live = (lane & 15) < cs.K - grp * 16;
    double* qx = a.data + cs.off_u + ENS_QX * arr + size_t(grp) * (Np * 16);
    double* qy = qx + (ENS_QY - ENS_QX) * arr;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int s = 4 * m + r;
            if (live && 4 * s + rg < Np) {
                qx[unsigned(64 * s + lane)] = in.m[0] * ar[m][r] + in.m[2] * as[m][r] - lx[m][r];
                qy[unsigned(64 * s + lane)] = in.m[1] * ar[m][r] + in.m[3] * as[m][r] - ly[m][r];
            }
        }
}

// B operands of one group's right-hand side: the flux differences at the face points for the lift, and for the volume
// products -Fr = -(rx Fx + ry Fy), -Fs = -(sx Fx + sy Fy), F = a u - nu q (negated so that the volume and lift products
// share one accumulator); and u at the nodes for the update.
template <int N>
struct EnsRhsIn {
    double u[ens_mfma_ks(N)], fr[ens_mfma_ks(N)], fs[ens_mfma_ks(N)], gb[N + 1];
};

template <int N>
__device__ __forceinline__ void ens_rhs_load(const EnsArgs& a, const EnsCase& cs, int grp, int lane, EnsRhsIn<N>& in) {
    constexpr int Np = ens_np(N), KS = ens_mfma_ks(N);
    const int left = cs.K - grp * 16, c0 = lane & 15, col = c0 < left ? c0 : left - 1, rg = lane >> 4;
    const size_t arr = size_t(cs.Kp) * Np;
    const double* u = a.data + cs.off_u + size_t(a.cur) * arr;
    const size_t to_x = (ENS_QX - a.cur) * arr, to_y = (ENS_QY - a.cur) * arr;
    const double* ug = u + size_t(grp) * (Np * 16);
    const double* g = a.geo + cs.off_geo + grp * 16;
    EnsLane<N> L;
    ens_lane<N>(a, cs, u, grp, col, rg, L);
    double um[N + 1], qm[N + 1], ym[N + 1], qx[KS], qy[KS], m[4];
#pragma unroll
    for (int k = 0; k <= N; ++k) {
        um[k] = ug[L.own[k]];
        qm[k] = (ug + to_x)[L.own[k]];
        ym[k] = (ug + to_y)[L.own[k]];
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        const unsigned at = 64 * s + 16 * rg + col;
        const bool in_range = 4 * s + rg < Np;
        in.u[s] = in_range ? ug[at] : 0.0;
        qx[s] = in_range ? (ug + to_x)[at] : 0.0;
        qy[s] = in_range ? (ug + to_y)[at] : 0.0;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) m[i] = (g + size_t(i) * cs.Kp)[unsigned(col)];
    __builtin_amdgcn_sched_barrier(0);   // the connectivity has been on its way longest: now the neighbours' values
#pragma unroll
    for (int k = 0; k <= N; ++k) qm[k] = L.nx * qm[k] + L.ny * ym[k];
    double up[N + 1], xp[N + 1], yp[N + 1];
#pragma unroll
    for (int k = 0; k <= N; ++k) {
        up[k] = L.up[L.nbr[k]];
        xp[k] = (L.up + to_x)[L.nbr[k]];
        yp[k] = (L.up + to_y)[L.nbr[k]];
    }
    __builtin_amdgcn_sched_barrier(0);
    const double ax = cs.ax, ay = cs.ay, nu = cs.nu;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        const double Fx = ax * in.u[s] - nu * qx[s], Fy = ay * in.u[s] - nu * qy[s];
        in.fr[s] = -(m[0] * Fx + m[1] * Fy);
        in.fs[s] = -(m[2] * Fx + m[3] * Fy);
    }
    const double an = ax * L.nx + ay * L.ny;
#pragma unroll
    for (int k = 0; k <= N; ++k) {
        const double qp = L.nx * xp[k] + L.ny * yp[k];
        const double fadv = an >= 0.0 ? an * um[k] : an * up[k];
        const double qhat = (L.own_side ? qp : qm[k]) - L.tf * (um[k] - up[k]);
        in.gb[k] = L.fs * ((an * um[k] - nu * qm[k]) - (fadv - nu * qhat));
    }
    __builtin_amdgcn_sched_barrier(0);
}

template <int N, bool UPDATE>
__device__ __forceinline__ void ens_rhs_mfma(const EnsArgs& a, const EnsCase& cs, const double* ops, int grp, int lane,
                                             const EnsRhsIn<N>& in) {
    constexpr int Np = ens_np(N), Nfp = N + 1;
    constexpr int MT = ens_mfma_mt(N), KS = ens_mfma_ks(N);
    const int rg = lane >> 4;
    const bool live = (lane & 15) < cs.K - grp * 16;
    const size_t arr = size_t(cs.Kp) * Np;
    double* base = a.data + cs.off_u + size_t(grp) * (Np * 16);
    double* res = base + ENS_RES * arr;
    const double* DrF = ops;
    const double* DsF = ops + MT * KS * 64;
    const double* LF = ops + 2 * MT * KS * 64;
    double old[KS];
    if constexpr (UPDATE) {   // in flight under the products
        const bool has = live && a.rk_a != 0.0;   // the first stage (a = 0) does not read res, so it needs no clearing
#pragma unroll
        for (int s = 0; s < KS; ++s) old[s] = has && 4 * s + rg < Np ? res[unsigned(64 * s + lane)] : 0.0;
    }
    d4_t acc[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = d4_t{0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < Nfp; ++k)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[m] = mfma64(LF[(m * Nfp + k) * 64 + lane], in.gb[k], acc[m]);
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            acc[m] = mfma64(DrF[(m * KS + s) * 64 + lane], in.fr[s], acc[m]);
            acc[m] = mfma64(DsF[(m * KS + s) * 64 + lane], in.fs[s], acc[m]);
        }
    const double dt = cs.dt;
    double* un = base + size_t(a.cur ^ 1) * arr;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        if (live && 4 * s + rg < Np) {
            const unsigned at = 64 * s + lane;
            const double rhs = acc[s / 4][s % 4];
            if constexpr (UPDATE) {
                const double rn = a.rk_a * old[s] + dt * rhs;
                res[at] = rn;
                un[at] = in.u[s] + a.rk_b * rn;
            } else {
                res[at] = rhs;
            }
        }
    }
}

template <int N, int P>
__device__ void ens_q_item(const EnsArgs& a, const EnsCase& cs, const double* ops, int blk, int p, int lane) {
    constexpr int Np = ens_np(N), Nfp = N + 1, R = ens_rows(N, P);
    const int Kp = cs.Kp;
    const int e0 = blk * kEnsLanes + lane;
    const bool live = e0 < cs.K;
    const int e = live ? e0 : cs.K - 1;
    const size_t arr = size_t(Kp) * Np;
    const double* __restrict__ u = a.data + cs.off_u + size_t(a.cur) * arr;
    double* __restrict__ qx = a.data + cs.off_u + ENS_QX * arr;
    double* __restrict__ qy = a.data + cs.off_u + ENS_QY * arr;
    const double* __restrict__ g = a.geo + cs.off_geo;
    const int* __restrict__ cn = a.conn + cs.off_conn;
    const int i0 = p * R;
    const double* __restrict__ DrT = ops + i0;                      // DrT[j * kEnsRows + i]
    const double* __restrict__ DsT = DrT + Np * kEnsRows;
    const double* __restrict__ LfT = DsT + Np * kEnsRows;           // LIFT^T[(f Nfp + k) * kEnsRows + i]
    double ar[R], as[R];
#pragma unroll
    for (int r = 0; r < R; ++r) ar[r] = as[r] = 0.0;
    // columns in chunks whose loads are all issued before the chunk's arithmetic (latency hiding)
    constexpr int CH = Np < 16 ? 4 : 8;
#pragma unroll 1
    for (int j0 = 0; j0 < Np; j0 += CH) {
        double uv[CH];
#pragma unroll
        for (int c = 0; c < CH; ++c) uv[c] = j0 + c < Np ? u[nidx(e, j0 + c, Np)] : 0.0;
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            if (j0 + c >= Np) break;
            const int j = j0 + c;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                ar[r] += DrT[j * kEnsRows + r] * uv[c];
                as[r] += DsT[j * kEnsRows + r] * uv[c];
            }
        }
    }
    const double rx = g[0 * Kp + e], ry = g[1 * Kp + e], sx = g[2 * Kp + e], sy = g[3 * Kp + e];
    double ox[R], oy[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        ox[r] = rx * ar[r] + sx * as[r];
        oy[r] = ry * ar[r] + sy * as[r];
    }
#pragma unroll 1
    for (int f = 0; f < 3; ++f) {
        const int c = cn[f * Kp + e];
        const int en = c >> 3, fn = (c >> 1) & 3;
        const bool own_side = c & 1;   // u^ = u-: no jump term
        const double nx = g[(4 + 4 * f) * Kp + e], ny = g[(5 + 4 * f) * Kp + e], fs = g[(6 + 4 * f) * Kp + e];
        double um[Nfp], up[Nfp];
#pragma unroll
        for (int k = 0; k < Nfp; ++k) {
            um[k] = u[nidx(e, face_node<N>(f, k), Np)];
            up[k] = u[nidx(en, face_node<N>(fn, N - k), Np)];
        }
#pragma unroll
        for (int k = 0; k < Nfp; ++k) {
            const double d = own_side ? 0.0 : fs * (um[k] - up[k]);
            const double gx = nx * d, gy = ny * d;
            const double* __restrict__ l = LfT + (f * Nfp + k) * kEnsRows;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                ox[r] -= l[r] * gx;
                oy[r] -= l[r] * gy;
            }
        }
    }
    if (live) {
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (i0 + r < Np) {
                qx[nidx(e0, i0 + r, Np)] = ox[r];
                qy[nidx(e0, i0 + r, Np)] = oy[r];
            }
    }
}

template <int N, int P>
__device__ void ens_rhs_item(const EnsArgs& a, const EnsCase& cs, const double* ops, int blk, int p, int lane) {
    constexpr int Np = ens_np(N), Nfp = N + 1, R = ens_rows(N, P);
    const int Kp = cs.Kp;
    const int e0 = blk * kEnsLanes + lane;
    const bool live = e0 < cs.K;
    const int e = live ? e0 : cs.K - 1;
    const size_t arr = size_t(Kp) * Np;
    double* __restrict__ base = a.data + cs.off_u;
    const double* __restrict__ u = base + size_t(a.cur) * arr;
    double* __restrict__ un = base + size_t(a.cur ^ 1) * arr;
    double* __restrict__ res = base + ENS_RES * arr;
    const double* __restrict__ qx = base + ENS_QX * arr;
    const double* __restrict__ qy = base + ENS_QY * arr;
    const double* __restrict__ g = a.geo + cs.off_geo;
    const int* __restrict__ cn = a.conn + cs.off_conn;
    const double ax = cs.ax, ay = cs.ay, nu = cs.nu;
    const int i0 = p * R;
    const double* __restrict__ DrT = ops + i0;
    const double* __restrict__ DsT = DrT + Np * kEnsRows;
    const double* __restrict__ LfT = DsT + Np * kEnsRows;
    const double rx = g[0 * Kp + e], ry = g[1 * Kp + e], sx = g[2 * Kp + e], sy = g[3 * Kp + e];
    double acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.0;
    // volume: -Dr (rx Fx + ry Fy) - Ds (sx Fx + sy Fy), F = a u - nu q
    constexpr int CH = Np < 4 ? Np : 4;
#pragma unroll 1
    for (int j0 = 0; j0 < Np; j0 += CH) {
        double uv[CH], xv[CH], yv[CH];
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const size_t id = nidx(e, j0 + c < Np ? j0 + c : Np - 1, Np);
            uv[c] = u[id];
            xv[c] = qx[id];
            yv[c] = qy[id];
        }
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            if (j0 + c >= Np) break;
            const int j = j0 + c;
            const double Fx = ax * uv[c] - nu * xv[c], Fy = ay * uv[c] - nu * yv[c];
            const double Fr = rx * Fx + ry * Fy, Fs = sx * Fx + sy * Fy;
#pragma unroll
            for (int r = 0; r < R; ++r) acc[r] -= DrT[j * kEnsRows + r] * Fr + DsT[j * kEnsRows + r] * Fs;
        }
    }
    // faces: LIFT(fscale ((a.n u- - nu n.q-) - ((a.n u)^ - nu n.q^)))
#pragma unroll 1
    for (int f = 0; f < 3; ++f) {
        const int c = cn[f * Kp + e];
        const int en = c >> 3, fn = (c >> 1) & 3;
        const bool own_side = c & 1;   // u^ = u-, so q^ = q+
        const double nx = g[(4 + 4 * f) * Kp + e], ny = g[(5 + 4 * f) * Kp + e];
        const double fs = g[(6 + 4 * f) * Kp + e], tf = g[(7 + 4 * f) * Kp + e];
        const double an = ax * nx + ay * ny;
        constexpr int KC = Nfp < 5 ? Nfp : 5;   // face points per batch of loads
#pragma unroll 1
        for (int k0 = 0; k0 < Nfp; k0 += KC) {
            double bu[KC], bq[KC], cu[KC], cq[KC];
#pragma unroll
            for (int t = 0; t < KC; ++t) {
                const int kk = k0 + t < Nfp ? k0 + t : Nfp - 1;
                const size_t im = nidx(e, face_node<N>(f, kk), Np);
                const size_t ip = nidx(en, face_node<N>(fn, N - kk), Np);
                bu[t] = u[im];
                bq[t] = nx * qx[im] + ny * qy[im];
                cu[t] = u[ip];
                cq[t] = nx * qx[ip] + ny * qy[ip];
            }
#pragma unroll
            for (int t = 0; t < KC; ++t) {
            const int k = k0 + t;
            if (k >= Nfp) break;
            const double um = bu[t], up = cu[t];
            const double qnm = bq[t], qnp = cq[t];
            const double fadv = an >= 0.0 ? an * um : an * up;
            const double qhat = (own_side ? qnp : qnm) - tf * (um - up);
            const double d = fs * ((an * um - nu * qnm) - (fadv - nu * qhat));
            const double* __restrict__ l = LfT + (f * Nfp + k) * kEnsRows;
#pragma unroll
            for (int r = 0; r < R; ++r) acc[r] += l[r] * d;
            }
        }
    }
    if (!live) return;
    const double dt = cs.dt;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if (i0 + r >= Np) continue;
        const size_t id = nidx(e0, i0 + r, Np);
        if (a.mode == 0) {
            res[id] = acc[r];
        } else {
            // the first stage (a = 0) does not read res, so it needs no clearing
            const double rn = (a.rk_a == 0.0 ? 0.0 : a.rk_a * res[id]) + dt * acc[r];
            res[id] = rn;
            un[id] = u[id] + a.rk_b * rn;
        }
    }
}

// MFMA variant: items are runs of at most kEnsWaves groups of 16 elements, one group per wave.  The fragments travel to
// LDS by DMA while the waves request their first group's inputs.  PASS 0: q; 1: right-hand side and stage update;
// 2: right-hand side into res.
template <int PASS, int N>
__global__ __launch_bounds__(64 * kEnsWaves) void ens_mfma_kernel(EnsArgs a) {
    constexpr size_t kBytes =
        size_t(2 * ens_mfma_mt(N) * ens_mfma_ks(N) + ens_mfma_mt(N) * ens_mfma_ksl(N)) * 64 * sizeof(double);
    __shared__ __attribute__((aligned(16))) double sop[dma_span(kBytes) / sizeof(double)];
    dma_stage_to_lds<kBytes>(sop, a.opsM[N]);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int xcd = blockIdx.x & 7, nbx = gridDim.x >> 3, bx = blockIdx.x >> 3;
    const int lo = a.chunk[xcd] + bx, hi = a.chunk[xcd + 1];
    std::conditional_t<PASS == 0, EnsQIn<N>, EnsRhsIn<N>> in;
    EnsCase cs;
    int grp = 0;
    // the wave's group of item it, its inputs on their way (false: no group; the same in all lanes)
    auto request = [&](int it) {
        const EnsItem item = a.items[it];
        cs = a.cases[item.c];
        grp = item.b0 + wave;
        const bool work = wave < item.nb && grp * 16 < cs.K;
        if (work) {
            if constexpr (PASS == 0) ens_q_load<N>(a, cs, grp, lane, in);
            else ens_rhs_load<N>(a, cs, grp, lane, in);
        }
        return work;
    };
    // whole waves only: a matrix instruction must not run with lanes left behind by the stores of the last group
    auto finish = [&]() {
        if constexpr (PASS == 0) ens_q_mfma<N>(a, cs, sop, grp, lane, in);
        else ens_rhs_mfma<N, PASS == 1>(a, cs, sop, grp, lane, in);
        __builtin_amdgcn_wave_barrier();
    };
    const bool first = lo < hi && request(lo);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's share of the fragments has landed
    __syncthreads();
    if (first) finish();
    for (int it = lo + nbx; it < hi; it += nbx)
        if (request(it)) finish();
}

// One persistent kernel per (pass, order, split) over that order's items: each is register-allocated for its
// own shape.  The order's operators are copied into LDS once per workgroup.
template <int PASS, int N, int P>
__global__ __launch_bounds__(64 * kEnsWaves) __attribute__((amdgpu_waves_per_eu(4))) void ens_kernel(EnsArgs a) {
    constexpr int nop = (2 * ens_np(N) + 3 * (N + 1)) * kEnsRows;
    __shared__ double sop[nop];
    for (int i = threadIdx.x; i < nop; i += 64 * kEnsWaves) sop[i] = a.ops[N][i];
    __syncthreads();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int xcd = blockIdx.x & 7, nbx = gridDim.x >> 3, bx = blockIdx.x >> 3;
    const int lo = a.chunk[xcd], hi = a.chunk[xcd + 1];
    for (int it = lo + bx; it < hi; it += nbx) {
        const EnsItem item = a.items[it];
        const EnsCase cs = a.cases[item.c];
        const int nblk = cs.Kp / kEnsLanes;
        for (int t = wave; t < item.nb * P; t += kEnsWaves) {
            const int blk = item.b0 + t / P, p = t % P;
            if (blk >= nblk) break;
            if constexpr (PASS == 0) ens_q_item<N, P>(a, cs, sop, blk, p, lane);
            else ens_rhs_item<N, P>(a, cs, sop, blk, p, lane);
        }
    }
}

template <int PASS, int N, int P>
static hipError_t launch_np(const EnsArgs& a, int grid, hipStream_t s) {
    if constexpr (ens_split_ok(N, P)) {
        hipLaunchKernelGGL((ens_kernel<PASS, N, P>), dim3(grid), dim3(64 * kEnsWaves), 0, s, a);
        return hipGetLastError();
    }
    return hipErrorInvalidValue;
}

template <int PASS, int N>
static hipError_t launch_n(int P, const EnsArgs& a, int grid, hipStream_t s) {
    if constexpr (N >= 2) {
        if (P == kEnsMfma) {
            if (PASS == 1 && a.mode == 0)
                hipLaunchKernelGGL((ens_mfma_kernel<PASS == 1 ? 2 : 0, N>), dim3(grid), dim3(64 * kEnsWaves), 0, s, a);
            else
                hipLaunchKernelGGL((ens_mfma_kernel<PASS, N>), dim3(grid), dim3(64 * kEnsWaves), 0, s, a);
            return hipGetLastError();
        }
    }
    switch (P) {
        case 1: return launch_np<PASS, N, 1>(a, grid, s);
        case 2: return launch_np<PASS, N, 2>(a, grid, s);
        case 4: return launch_np<PASS, N, 4>(a, grid, s);
        case 8: return launch_np<PASS, N, 8>(a, grid, s);
        default: return hipErrorInvalidValue;
    }
}

template <int PASS>
static hipError_t launch_pass(int N, int P, const EnsArgs& a, int grid, hipStream_t s) {
    switch (N) {
        case 1: return launch_n<PASS, 1>(P, a, grid, s);
        case 2: return launch_n<PASS, 2>(P, a, grid, s);
        case 3: return launch_n<PASS, 3>(P, a, grid, s);
        case 4: return launch_n<PASS, 4>(P, a, grid, s);
        case 5: return launch_n<PASS, 5>(P, a, grid, s);
        case 6: return launch_n<PASS, 6>(P, a, grid, s);
        case 7: return launch_n<PASS, 7>(P, a, grid, s);
        case 8: return launch_n<PASS, 8>(P, a, grid, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_ens_q(int N, int P, const EnsArgs& a, int grid, hipStream_t s) {
    return launch_pass<0>(N, P, a, grid, s);
}
hipError_t launch_ens_rhs(int N, int P, const EnsArgs& a, int grid, hipStream_t s) {
    return launch_pass<1>(N, P, a, grid, s);
}

// resident workgroups per CU: LDS (the order's operator table or MFMA fragments), and waves per SIMD: four, two for
// the MFMA kernels of orders 5 to 8 (more than 128 registers)
int ens_blocks_per_cu(int N, int P) {
    const size_t lds = P == kEnsMfma
        ? size_t(2 * ens_mfma_mt(N) * ens_mfma_ks(N) + ens_mfma_mt(N) * ens_mfma_ksl(N)) * 64 * sizeof(double)
        : size_t(2 * ens_np(N) + 3 * (N + 1)) * kEnsRows * sizeof(double);
    const int by_lds = int((160u * 1024u) / lds);
    const int by_waves = (P == kEnsMfma && N >= 5 ? 8 : 16) / kEnsWaves;
    const int b = by_lds < by_waves ? by_lds : by_waves;
    return b > 0 ? b : 1;
}

}  // namespace dg
