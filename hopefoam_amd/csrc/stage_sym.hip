// FP64 right-hand side + stage update on the mirror-symmetric halves of the reference-element operators, gfx950.
//
// The same weak form as stage_kernels.hip, one wavefront per 16 elements, with the contractions cut in half by the
// reflection r <-> s of the reference triangle (a prime marks the mirror node or point):
//   interpolation  q(p), q(p') = Qe(p) +- Qo(p),  Qe = Ve (q_a + q_a'), Qo = Vo (q_a - q_a')
//   projection     rhs_a, rhs_a' = E +- O with
//                  E = sum_p 1/2 (Pr[a,p] + Pr[a',p]) (Fr(p) + Fs(p')),
//                  O = sum_p 1/2 (Pr[a,p] - Pr[a',p]) (Fr(p) - Fs(p'))      (since Ps[a,p] = Pr[a',p'])
//   lift           faces 0 and 2 are each other's mirror images: their fluxes enter as sum and difference.
// Nothing is assumed of the element's shape: Fr, Fs are the contravariant fluxes at the points, whatever the
// geometric factors are.  A fixed node is a row whose "pair" is the node twice (its difference is 0, its sum twice
// the value, with half the operator entry), so no lane branches.
//
// Why: on gfx950 f64 MFMA (64 clk each) and f64 VALU instructions do not overlap, neither in one wavefront nor
// between the wavefronts of a SIMD, so their times add.  At N = 6 the halves take 324 MFMA per group of 16 elements
// instead of 600 for about 200 more additions.  Two wavefronts per SIMD (256 registers, N <= 6) hide most of the gathers
// and the dependent chains; an f64 FMA then issues every 4.3 clk instead of 5.6.
// Account of the some 44,000 clk that a SIMD has per group at N = 6, K = 131072 (163 to 169 us at 2.1 GHz): 20,700 of
// matrix products, 8,600 of 2,000 f64 VALU instructions, about 5,000 of 1,200 other VALU instructions.  The other 10,000
// are waits that the second wavefront does not cover (the counters name memory: 17 % of the wavefronts' time) and LDS,
// scalar and branch issue, which they do not tell apart.
// Measured (us per stage; before: whole operators, one wavefront per SIMD, own traces by lane shuffles):
//   LF, K = 131072:  N = 2  49.4 -> 40.4   3  87.0 -> 71.0   4  119 -> 92.5   5  200 -> 127   6  237 -> 163
//   LF, K = 32768:   N = 7  185 -> 73      8  228 -> 110 (112 since its first stage reads, its last writes no residual)
//   Roe, K = 131072: N = 2  58.5 -> 44.3   3  103.8 -> 78.4  4  137 -> 98.5
//   small meshes:    N = 4 Roe, K = 1024  20.7 -> 14.2;  N = 4 advection, K = 2048  8.9 -> 6.2
// Order 1 takes the whole operators in this kernel's layout (SymDims::whole): its 3 nodes fill one tile either way, and
// on the halves large meshes were slower than before (LF: 35.0 -> 36.5 us at K = 131072, 15.0 -> 19.6 at 45000).  Before,
// on the halves, now:  LF, K = 131072 35.0, 36.5, 30.3;  45000 15.0, 19.6, 12.6;  32768 11.5, 12.1, 9.6;  8192 8.2, 6.8,
// 5.5;  Roe, K = 131072 43.6, 40.3, 34.4;  advection, K = 524288 39.0, 43.0, 36.7
//
// Layout: K step s of the interpolation takes node row 4 s + rg from row group rg; with the f64 accumulator map
// (register r of row group rg holds row 4 r + rg) that is also the row of accumulator register r of tile m for
// s = 4 m + r, so a lane updates the nodes it loaded.  Likewise point row 16 t + 4 r + rg of tile t is the lane's
// own operand of projection step 4 t + r.
#include <hip/hip_runtime.h>

#include "dg_common.hpp"
#include "lds_stage.hpp"
#include "stage_device.hpp"
#include "stage_kernels.hpp"
#include "stage_sym.hpp"

namespace dg {

// Wavefronts per block, and per SIMD as asked of the register allocation: two per SIMD where the kernel fits 256
// registers without spilling, one beyond.  At K = 131072 and N = 6 two per SIMD take 163 us, one about 190 us; spilling
// (all face loads ahead of the volume work, both fluxes in one kernel, 64-bit lane addresses) cost more than the
// second wavefront gave, 229 to 305 us.
template <int N>
constexpr int sym_waves() { return N <= 2 || N >= 7 ? 4 : 8; }
template <int N>
constexpr int sym_per_simd() { return N <= 6 ? 2 : 1; }

// LDS of a block: the operator fragments and, where they fit beside them, one group's nodal values per wavefront (the
// volume, the own traces and the update all read them from there, so that no registers hold them; at order 8 they do
// not fit, at order 1 the three nodes per variable are registers' work)
template <int N, int NV>
struct SymLds {
    static constexpr size_t frag = dma_span(size_t(SymDims<N>::nF) * sizeof(double));
    static constexpr size_t nodes = dma_span(size_t(NV) * SymDims<N>::Np * 16 * sizeof(double));
    static constexpr bool hold = N >= 2 && frag + sym_waves<N>() * nodes <= 160 * 1024;
};

// Transposes a 4 x 4 matrix over the row groups: in: x[g] holds, in row group v, entry (g, v); out: x[v] holds, in
// row group g, entry (g, v).  v_permlane32_swap exchanges the upper half of its first operand with the lower half of
// its second, v_permlane16_swap the odd rows of 16 lanes with the even ones.
__device__ __forceinline__ void transpose_rows(double (&x)[4]) {
    unsigned w[4][2];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const unsigned long long u = __builtin_bit_cast(unsigned long long, x[g]);
        w[g][0] = unsigned(u);
        w[g][1] = unsigned(u >> 32);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const auto p = __builtin_amdgcn_permlane32_swap(w[0][h], w[2][h], false, false);
        const auto q = __builtin_amdgcn_permlane32_swap(w[1][h], w[3][h], false, false);
        const auto r = __builtin_amdgcn_permlane16_swap(p[0], q[0], false, false);
        const auto s = __builtin_amdgcn_permlane16_swap(p[1], q[1], false, false);
        w[0][h] = r[0];
        w[1][h] = r[1];
        w[2][h] = s[0];
        w[3][h] = s[1];
    }
#pragma unroll
    for (int v = 0; v < 4; ++v)
        x[v] = __builtin_bit_cast(double, (unsigned long long)(w[v][1]) << 32 | w[v][0]);
}

// UPDATE: the fused stage update (mode 1), else the right-hand side (mode 0).  The flux and the mode are template
// parameters: with both fluxes in one kernel it spills.
template <int N, int PHYS, int FLUX, bool UPDATE>
__global__ __launch_bounds__(64 * sym_waves<N>(), sym_per_simd<N>()) void stage_sym_kernel(StageArgs a) {
    using D = SymDims<N>;
    using VF = VolumeFlux<PHYS, double>;
    constexpr int NV = VF::NV, Np = D::Np, Nfp = D::Nfp, Nfq = D::Nfq, SF = D::SF;
    constexpr int KE = D::KE, KO = D::KO, ME = D::ME, MO = D::MO;
    constexpr int KOA = KO ? KO : 1, MOA = MO ? MO : 1;   // array lengths
    constexpr int WPB = sym_waves<N>();
    constexpr size_t GS = size_t(NV) * Np * 16;
    constexpr size_t kFrBytes = size_t(D::nF) * sizeof(double);
    using S = SymLds<N, NV>;
    constexpr bool kLds = S::hold, kEarly = N <= 2;

    __shared__ __attribute__((aligned(16))) double frag[S::frag / sizeof(double)];
    __shared__ __attribute__((aligned(16))) double nodes[kLds ? WPB * S::nodes / sizeof(double) : 2];

    // the wavefront's number in a scalar register: a group's addresses are then a scalar base and one lane offset
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, rg = lane >> 4;
    const int K = a.K, groups = (K + 15) >> 4;
    // XCD-aware schedule: block b runs on XCD b % 8, each XCD walks a contiguous range of groups; the wavefronts of
    // a block take groups nbx apart, so that a small mesh spreads over the compute units first
    const int xcd = blockIdx.x & 7, nbx = gridDim.x >> 3, bx = blockIdx.x >> 3;
    const int g_lo = int((long long)groups * xcd / 8), g_hi = int((long long)groups * (xcd + 1) / 8);
    if (g_lo + bx >= g_hi) return;          // no group for this block
    const int gstride = nbx * WPB;
    int grp = g_lo + wave * nbx + bx;
    dma_stage_to_lds<kFrBytes>(frag, a.VqF);
    double* qw = nodes + (kLds ? wave * (S::nodes / sizeof(double)) : 0);   // the group's nodal values
    if (kLds && grp < g_hi) dma_to_lds_whole<GS * sizeof(double)>(a.q_in + size_t(grp) * GS, qw, lane);
    // the face interpolation matrix from the constant address space: its uniform reads are scalar loads
    typedef const __attribute__((address_space(4))) double cdouble;
    cdouble* Vf = reinterpret_cast<cdouble*>(reinterpret_cast<uintptr_t>(a.Vf));
    const double* __restrict__ geo = static_cast<const double*>(a.geo);
    const double* VE = frag;
    const double* VO = VE + D::TE * KE * 64;
    const double* P = frag + D::nV;
    const double* L = P + D::nP;

    // byte offsets of this lane's node pairs inside a variable's block of a group: unsigned, so that an access is a
    // scalar base plus one 32-bit lane offset
    unsigned na[KE], nb[KOA];
#pragma unroll
    for (int s = 0; s < KE; ++s) {
        const unsigned ab = unsigned(a.rows[4 * s + rg]);
        na[s] = ((ab & 255u) * 16 + col) * 8;
        if (s < KO) nb[s < KO ? s : 0] = ((ab >> 8) * 16 + col) * 8;
    }
    auto load_nodes = [&](const double* src, double (&x)[NV][KE], double (&y)[NV][KOA]) {
#pragma unroll
        for (int v = 0; v < NV; ++v)
#pragma unroll
            for (int s = 0; s < KE; ++s) {
                x[v][s] = at_lane(src + v * Np * 16, na[s]);
                if (s < KO) y[v][s < KO ? s : 0] = at_lane(src + v * Np * 16, nb[s < KO ? s : 0]);
            }
    };
    auto load_old = [&](const double* src, double (&x)[NV][KE], double (&y)[NV][KOA]) {
        if (a.res_in) {
            load_nodes(src, x, y);
        } else {
#pragma unroll
            for (int v = 0; v < NV; ++v)
#pragma unroll
                for (int s = 0; s < KE; ++s) {
                    x[v][s] = 0.0;
                    if (s < KO) y[v][s < KO ? s : 0] = 0.0;
                }
        }
    };
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the fragments and the first group have landed
    __syncthreads();

    for (; grp < g_hi; grp += gstride) {
        const int e = grp * 16 + col < K ? grp * 16 + col : K - 1;
        const double* __restrict__ qg = a.q_in + size_t(grp) * GS;
        double* out_g = a.q_out + size_t(grp) * GS;
        double* res_g = a.res + size_t(grp) * GS;
        const double* old_g = a.res_in + size_t(grp) * GS;
        const double* qn = kLds ? qw : qg;
        // sums and differences of the node pairs: kept in registers, or formed from LDS for every point tile
        double qe[kLds ? 1 : NV][KE], qo[kLds ? 1 : NV][KOA];
        if constexpr (!kLds) {
            double xa[NV][KE], xb[NV][KOA];
            load_nodes(qg, xa, xb);
#pragma unroll
            for (int v = 0; v < NV; ++v)
#pragma unroll
                for (int s = 0; s < KE; ++s) {
                    const int so = s < KO ? s : 0;
                    qe[v][s] = D::whole ? xa[v][s] : xa[v][s] + (s < KO ? xb[v][so] : xa[v][s]);
                    if (s < KO) qo[v][so] = xa[v][s] - xb[v][so];
                }
        }
        int cn[3];
#pragma unroll
        for (int f = 0; f < 3; ++f) cn[f] = a.conn[f * K + e];
        const double rx = geo[G_RX * K + e], ry = geo[G_RY * K + e], sx = geo[G_SX * K + e], sy = geo[G_SY * K + e];

        auto face_geo = [&](int f, double& nx, double& ny, double& fsc) {
            nx = geo[(G_NX0 + 3 * f) * K + e];
            ny = geo[(G_NY0 + 3 * f) * K + e];
            fsc = geo[(G_FS0 + 3 * f) * K + e];
        };
        auto load_face = [&](int f, double (&own)[Nfp], double (&oth)[Nfp]) {   // lane (col, rg): variable rg
            const int v = rg < NV ? rg : 0;
            const bool keep = gather_face<N, NV>(a, cn[f], f, e, rg, oth);
#pragma unroll
            for (int k = 0; k < Nfp; ++k) own[k] = qn[(v * Np + face_node<N>(f, k)) * 16 + col];
            return keep;
        };
        // small orders: the faces' nodes and the residual are requested here and arrive behind the volume work; beyond,
        // they would spill and the SIMD's other wavefront hides them
        double own0[Nfp], oth0[Nfp], own1[Nfp], oth1[Nfp], own2[Nfp], oth2[Nfp], nx0, ny0, fs0, nx1, ny1, fs1, nx2, ny2, fs2;
        bool keep0, keep1, keep2;
        double ra[NV][KE], rb[NV][KOA], ua[NV][KE], ub[NV][KOA];
        if constexpr (kEarly) {
            keep0 = load_face(0, own0, oth0);
            keep2 = load_face(2, own2, oth2);
            face_geo(0, nx0, ny0, fs0);
            face_geo(2, nx2, ny2, fs2);
            keep1 = load_face(1, own1, oth1);
            face_geo(1, nx1, ny1, fs1);
            if constexpr (UPDATE) load_old(old_g, ra, rb);
        }

        d4_t accE[NV][ME], accO[NV][MOA];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
#pragma unroll
            for (int m = 0; m < ME; ++m) accE[v][m] = d4_t{0, 0, 0, 0};
#pragma unroll
            for (int m = 0; m < MO; ++m) accO[v][m] = d4_t{0, 0, 0, 0};
        }

        // ---- volume
#pragma unroll
        for (int t = 0; t < D::TE; ++t) {
            d4_t ce[NV], co[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) ce[v] = co[v] = d4_t{0, 0, 0, 0};
            if constexpr (kLds) {   // read the nodes again for every tile: held in registers they would spill
#pragma unroll
                for (int s = 0; s < KE; ++s) {
                    asm volatile("" : "+v"(na[s]));
                    if (s < KO) asm volatile("" : "+v"(nb[s < KO ? s : 0]));
                }
            }
#pragma unroll
            for (int s = 0; s < KE; ++s) {
                const int so = s < KO ? s : 0;
                const double Ae = VE[(t * KE + s) * 64 + lane];
                const double Ao = t < D::TO && s < KO ? VO[(t * KO + so) * 64 + lane] : 0.0;
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    double be, bo;
                    if constexpr (kLds) {
                        const double x = at_lane(qw + v * Np * 16, na[s]), y = s < KO ? at_lane(qw + v * Np * 16, nb[so]) : x;
                        be = D::whole ? x : x + y;
                        bo = x - y;
                    } else {
                        be = qe[v][s];
                        bo = qo[v][so];
                    }
                    ce[v] = mfma4(Ae, be, ce[v]);
                    if (t < D::TO && s < KO) co[v] = mfma4(Ao, bo, co[v]);
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int ks = 4 * t + r;
                if (ks >= D::KT) continue;
                // point rows past the last (in the last step only) have zero operator columns, but the flux of their
                // zero state is not finite
                const bool pad = 4 * ks + 3 >= D::qrow && 4 * ks + rg >= D::qrow;
                double q1[NV], fr1[NV], fs1[NV];
                if constexpr (D::whole) {
#pragma unroll
                    for (int v = 0; v < NV; ++v) q1[v] = ce[v][r];
                    VF::eval(q1, a.ax, a.ay, a.gamma, rx, ry, sx, sy, fr1, fs1);
                    const double* A = P + size_t(2 * ks) * ME * 64 + lane;
#pragma unroll
                    for (int v = 0; v < NV; ++v) {
                        if (pad) fr1[v] = fs1[v] = 0.0;
#pragma unroll
                        for (int m = 0; m < ME; ++m) accE[v][m] = mfma4(A[m * 64], fr1[v], accE[v][m]);
#pragma unroll
                        for (int m = 0; m < ME; ++m) accE[v][m] = mfma4(A[(ME + m) * 64], fs1[v], accE[v][m]);
                    }
                } else if (ks < D::KP) {
                    double q2[NV], fr2[NV], fs2[NV];
#pragma unroll
                    for (int v = 0; v < NV; ++v) {
                        q1[v] = ce[v][r] + co[v][r];
                        q2[v] = ce[v][r] - co[v][r];
                    }
                    VF::eval(q1, a.ax, a.ay, a.gamma, rx, ry, sx, sy, fr1, fs1);
                    VF::eval(q2, a.ax, a.ay, a.gamma, rx, ry, sx, sy, fr2, fs2);
                    const double* A = P + size_t(2 * ks) * (ME + MO) * 64 + lane;
#pragma unroll
                    for (int v = 0; v < NV; ++v) {
                        if (pad) fr1[v] = fs1[v] = fr2[v] = fs2[v] = 0.0;
                        const double s1 = fr1[v] + fs2[v], d1 = fr1[v] - fs2[v];
                        const double s2 = fr2[v] + fs1[v], d2 = fr2[v] - fs1[v];
#pragma unroll
                        for (int m = 0; m < ME; ++m) accE[v][m] = mfma4(A[m * 64], s1, accE[v][m]);
#pragma unroll
                        for (int m = 0; m < MO; ++m) accO[v][m] = mfma4(A[(ME + m) * 64], d1, accO[v][m]);
#pragma unroll
                        for (int m = 0; m < ME; ++m) accE[v][m] = mfma4(A[(ME + MO + m) * 64], s2, accE[v][m]);
#pragma unroll
                        for (int m = 0; m < MO; ++m) accO[v][m] = mfma4(A[(2 * ME + MO + m) * 64], d2, accO[v][m]);
                    }
                } else {
#pragma unroll
                    for (int v = 0; v < NV; ++v) q1[v] = ce[v][r];
                    VF::eval(q1, a.ax, a.ay, a.gamma, rx, ry, sx, sy, fr1, fs1);
                    const double* A = P + size_t(D::KP + ks) * (ME + MO) * 64 + lane;
#pragma unroll
                    for (int v = 0; v < NV; ++v) {
                        if (pad) fr1[v] = fs1[v] = 0.0;
                        const double s1 = fr1[v] + fs1[v], d1 = fr1[v] - fs1[v];
#pragma unroll
                        for (int m = 0; m < ME; ++m) accE[v][m] = mfma4(A[m * 64], s1, accE[v][m]);
#pragma unroll
                        for (int m = 0; m < MO; ++m) accO[v][m] = mfma4(A[(ME + m) * 64], d1, accO[v][m]);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);   // one step's fluxes live at a time
            }
        }
        if constexpr (!kEarly) __builtin_amdgcn_sched_barrier(0);   // the face loads stay behind the volume: ahead of it they spill

        // ---- faces 0 and 2 together (face 2 from its far end, so that a lane's items are mirror images), then face
        // 1.  Lane (col, rg) interpolates variable rg's own and outer nodes to four Gauss points at a time; a
        // transpose over the row groups hands them to the lane of Gauss point 4 j + rg, which forms the flux.
        // minus the scaled normal flux at Gauss point 4 j + rg (mirror: Nfq - 1 - (4 j + rg)) of face f
        auto face_flux = [&](int f, int j, bool mirror, const double (&own)[Nfp], const double (&oth)[Nfp], bool keep,
                             double nx, double ny, double fsc, double (&bf)[NV]) {
            double qM[4], qP[4], Fs[NV];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                qM[i] = qP[i] = 0.0;
                if (4 * j + i >= Nfq) continue;
                const int g = mirror ? Nfq - 1 - (4 * j + i) : 4 * j + i;
#pragma unroll
                for (int k = 0; k < Nfp; ++k) {
                    const double w = Vf[g * Nfp + k];
                    qM[i] += w * own[k];
                    qP[i] += w * oth[k];
                }
            }
            if constexpr (NV == 1) {   // every row group holds the one variable
                qM[0] = rg < 2 ? (rg == 0 ? qM[0] : qM[1]) : (rg == 2 ? qM[2] : qM[3]);
                qP[0] = rg < 2 ? (rg == 0 ? qP[0] : qP[1]) : (rg == 2 ? qP[2] : qP[3]);
            } else {
                transpose_rows(qM);
                transpose_rows(qP);
            }
            const bool copy_own = cn[f] < 0 && -cn[f] - 1 != BC_FIXED;
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                bf[v] = 0.0;
                qP[v] = copy_own ? qM[v] : (keep ? qP[v] : 0.0);
            }
            if (4 * j + rg < Nfq) {
                if constexpr (PHYS == PHYS_EULER) {
                    if (cn[f] < 0 && -cn[f] - 1 == BC_WALL) {   // mirror the momentum
                        const double mn = qP[1] * nx + qP[2] * ny;
                        qP[1] -= 2.0 * mn * nx;
                        qP[2] -= 2.0 * mn * ny;
                    }
                }
                if constexpr (PHYS == PHYS_ADVECT) {   // upwind, or the central "average" flux without the |vn| term
                    const double vn = nx * a.ax + ny * a.ay;
                    const double diss = a.flux == FLUX_AVERAGE ? 0.0 : fabs(vn);
                    Fs[0] = (vn * qM[0] + vn * qP[0]) * 0.5 + diss * (qM[0] - qP[0]) * 0.5;
                } else if constexpr (FLUX == FLUX_ROE) {
                    roe_flux<double>(a.gamma, nx, ny, qM, qP, Fs);
                } else {
                    llf_flux<double>(a.gamma, nx, ny, qM, qP, Fs);
                }
#pragma unroll
                for (int v = 0; v < NV; ++v) bf[v] = -fsc * Fs[v];
            }
        };
        {
            if constexpr (!kEarly) {
                keep0 = load_face(0, own0, oth0);
                keep2 = load_face(2, own2, oth2);
                face_geo(0, nx0, ny0, fs0);
                face_geo(2, nx2, ny2, fs2);
            }
#pragma unroll
            for (int j = 0; j < SF; ++j) {
                double b0[NV], b2[NV];
                face_flux(0, j, false, own0, oth0, keep0, nx0, ny0, fs0, b0);
                face_flux(2, j, !D::whole, own2, oth2, keep2, nx2, ny2, fs2, b2);
                const double* A = L + size_t(j) * (ME + MO) * 64 + lane;
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    if constexpr (D::whole) {
#pragma unroll
                        for (int m = 0; m < ME; ++m) accE[v][m] = mfma4(A[m * 64], b0[v], accE[v][m]);
#pragma unroll
                        for (int m = 0; m < ME; ++m) accE[v][m] = mfma4(A[(SF * ME + m) * 64], b2[v], accE[v][m]);
                        continue;
                    }
                    const double s = b0[v] + b2[v], d = b0[v] - b2[v];
#pragma unroll
                    for (int m = 0; m < ME; ++m) accE[v][m] = mfma4(A[m * 64], s, accE[v][m]);
#pragma unroll
                    for (int m = 0; m < MO; ++m) accO[v][m] = mfma4(A[(ME + m) * 64], d, accO[v][m]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        {
            if constexpr (!kEarly) {
                keep1 = load_face(1, own1, oth1);
                face_geo(1, nx1, ny1, fs1);
            }
#pragma unroll
            for (int j = 0; j < SF; ++j) {
                double b1[NV];
                face_flux(1, j, false, own1, oth1, keep1, nx1, ny1, fs1, b1);
                const double* A = L + size_t((D::whole ? 2 : 1) * SF + j) * (ME + MO) * 64 + lane;
#pragma unroll
                for (int v = 0; v < NV; ++v) {
#pragma unroll
                    for (int m = 0; m < ME; ++m) accE[v][m] = mfma4(A[m * 64], b1[v], accE[v][m]);
#pragma unroll
                    for (int m = 0; m < MO; ++m) accO[v][m] = mfma4(A[(ME + m) * 64], b1[v], accO[v][m]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }

        // ---- output: rows 4 s + rg, s = 4 m + r (padding columns keep evolving a copy of element K - 1).  Every load
        // comes before the first store (the compiler keeps loads behind stores that could alias).
        if constexpr (UPDATE) {
            if constexpr (!kEarly) load_old(old_g, ra, rb);
            load_nodes(qn, ua, ub);
        }
        if constexpr (kLds) {
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the reads of the buffer have returned
            if (grp + gstride < g_hi)
                dma_to_lds_whole<GS * sizeof(double)>(a.q_in + size_t(grp + gstride) * GS, qw, lane);
        }
        if constexpr (UPDATE) {
            if (a.mode == 2) {
#pragma unroll
                for (int v = 0; v < NV; ++v)
#pragma unroll
                    for (int s = 0; s < KE; ++s) {
                        ra[v][s] -= ua[v][s];
                        if (s < KO) rb[v][s < KO ? s : 0] -= ub[v][s < KO ? s : 0];
                    }
            }
        }
        // f(row set s of variable v, its even and odd part, whether this lane has row a, row b)
        auto rows = [&](auto f) {
#pragma unroll
            for (int v = 0; v < NV; ++v)
#pragma unroll
                for (int s = 0; s < KE; ++s) {
                    const int so = s < KO ? s : 0;
                    const double E = accE[v][s / 4][s % 4], O = s < KO ? accO[v][so / 4][s % 4] : 0.0;
                    const bool on = 4 * s + 3 < D::nrow || 4 * s + rg < D::nrow;
                    const bool pair = s < KO && (4 * s + 3 < D::npair || 4 * s + rg < D::npair);
                    f(v, s, so, E, O, on, pair);
                }
        };
        if constexpr (!UPDATE) {
            rows([&](int v, int s, int so, double E, double O, bool on, bool pair) {
                double* ov = out_g + v * Np * 16;
                if (on) put_lane(ov, na[s], E + O);
                if (pair) put_lane(ov, nb[so], E - O);
            });
        } else {
            rows([&](int v, int s, int so, double E, double O, bool, bool) {
                ra[v][s] = a.rk_a * ra[v][s] + a.dt * (E + O);
                if (s < KO) rb[v][so] = a.rk_a * rb[v][so] + a.dt * (E - O);
            });
            if (a.res)
                rows([&](int v, int s, int so, double, double, bool on, bool pair) {
                    double* rv = res_g + v * Np * 16;
                    if (on) put_lane(rv, na[s], ra[v][s]);
                    if (pair) put_lane(rv, nb[so], rb[v][so]);
                });
            rows([&](int v, int s, int so, double, double, bool on, bool pair) {
                double* ov = out_g + v * Np * 16;
                if (on) put_lane(ov, na[s], ua[v][s] + a.rk_b * ra[v][s]);
                if (pair) put_lane(ov, nb[so], ub[v][so] + a.rk_b * rb[v][so]);
            });
        }
        if constexpr (kLds) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the next group has landed
    }
}

template <int N, int PHYS, int FLUX, bool UPDATE>
static hipError_t launch_sym_inst(const StageArgs& a, int ncu, hipStream_t st) {
    constexpr int threads = 64 * sym_waves<N>();
    static int per_cu = 0;   // resident blocks per compute unit
    if (per_cu < 1) {
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, stage_sym_kernel<N, PHYS, FLUX, UPDATE>, threads, 0) !=
            hipSuccess)
            n = 1;
        per_cu = n < 1 ? 1 : n;
    }
    const int groups = (a.K + 15) / 16;
    // a persistent grid: a block per group up to one per compute unit, then one more for every compute unit as their
    // wavefronts fill (the wavefronts of a block take groups apart, so that with more blocks than that each leaves its last
    // SIMDs idle; as many as are resident -> as here, order 1 LF, K = 32768: 11.6 -> 9.6 us, order 2 Roe, K = 11834: 11.3
    // -> 8.0; with fewer some compute units hold a block more than the others: order 2 LF, K = 20174, 320 blocks 11.6, 512
    // 11.0, order 1 9.0 and 8.4)
    const int full = (groups + sym_waves<N>() - 1) / sym_waves<N>(), least = groups < ncu ? groups : ncu;
    const int even = full <= ncu ? full : (full + ncu - 1) / ncu * ncu;
    int nb = even < least ? least : even < ncu * per_cu ? even : ncu * per_cu;
    nb = nb < 8 ? 8 : (nb + 7) / 8 * 8;
    if (a.block_cap > 0 && nb > a.block_cap) nb = a.block_cap < 8 ? 8 : a.block_cap / 8 * 8;
    hipLaunchKernelGGL((stage_sym_kernel<N, PHYS, FLUX, UPDATE>), dim3(nb), dim3(threads), 0, st, a);
    return hipGetLastError();
}

template <int N, int PHYS, int FLUX>
static hipError_t launch_sym_flux(const StageArgs& a, int ncu, hipStream_t st) {
    return a.mode != 0 ? launch_sym_inst<N, PHYS, FLUX, true>(a, ncu, st)
                       : launch_sym_inst<N, PHYS, FLUX, false>(a, ncu, st);
}

template <int N>
static hipError_t launch_sym_n(int phys, const StageArgs& a, int ncu, hipStream_t st) {
    if (phys == PHYS_ADVECT) return launch_sym_flux<N, PHYS_ADVECT, FLUX_UPWIND>(a, ncu, st);
    return a.flux == FLUX_ROE ? launch_sym_flux<N, PHYS_EULER, FLUX_ROE>(a, ncu, st)
                              : launch_sym_flux<N, PHYS_EULER, FLUX_LF>(a, ncu, st);
}

hipError_t launch_stage_sym(int N, int phys, const StageArgs& a, int ncu, hipStream_t st) {
    switch (N) {
        case 1: return launch_sym_n<1>(phys, a, ncu, st);
        case 2: return launch_sym_n<2>(phys, a, ncu, st);
        case 3: return launch_sym_n<3>(phys, a, ncu, st);
        case 4: return launch_sym_n<4>(phys, a, ncu, st);
        case 5: return launch_sym_n<5>(phys, a, ncu, st);
        case 6: return launch_sym_n<6>(phys, a, ncu, st);
        case 7: return launch_sym_n<7>(phys, a, ncu, st);
        case 8: return launch_sym_n<8>(phys, a, ncu, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace dg
