// Device pieces shared by the stage kernels: the 16x16x4 MFMA wrappers, the physical and numerical fluxes, and the
// gather of a face's outer nodes.
#pragma once
#include <hip/hip_runtime.h>

#include "dg_common.hpp"
#include "stage_kernels.hpp"

namespace dg {

typedef double d4_t __attribute__((ext_vector_type(4)));
typedef float f4_t __attribute__((ext_vector_type(4)));

template <typename T>
struct Vec4;
template <>
struct Vec4<float> { typedef f4_t type; };

// Row of the 16x16 accumulator held in register r of a lane of row group rg (= lane / 16).
template <typename T>
struct RowMap {
    __host__ __device__ static constexpr int row(int rg, int r) { return dg::mfma_row<T>(rg, r); }
};

__device__ __forceinline__ d4_t mfma4(double a, double b, d4_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4_t mfma4(float a, float b, f4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Reciprocal and square root of the flux arithmetic.  FP64: v_rcp_f64 refined by two Newton steps r += r (1 - x r) in
// fused multiply-adds (each step squares the relative error, so the result is within an ulp of 1 / x), five instructions
// instead of the eleven of an IEEE division (the densities it is taken of are positive and normal); v_rsq_f64 refined
// by one coupled step for sqrt(x) and 1 / (2 sqrt(x)) and two residual corrections g += h (x - g g), within an ulp of
// sqrt(x), in half the instructions of the scaled library square root (0 and infinity come out as themselves, a negative
// number as NaN).  The residual x - g g of a subnormal x is rounded to a multiple of the least number: 0, as it should be.
// FP32: the hardware's v_rcp_f32 / v_sqrt_f32 (about 1 ulp), far below the FP32 and bf16x3 paths' contraction
// round-off, in one instruction instead of the ten of an IEEE division or square root.
__device__ __forceinline__ double inv(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = fma(fma(-x, r, 1.0), r, r);
    return fma(fma(-x, r, 1.0), r, r);
}
__device__ __forceinline__ float inv(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ double fsqrt(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double r = fma(-h, g, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
    g = fma(fma(-g, g, x), h, g);
    g = fma(fma(-g, g, x), h, g);
    return __builtin_amdgcn_class(x, 0x260) ? x : g;   // -0, +0, +inf
}
__device__ __forceinline__ float fsqrt(float x) { return __builtin_amdgcn_sqrtf(x); }

// ---------------------------------------------------------------- physics
template <int PHYS, typename T>
struct VolumeFlux;

template <typename T>
struct VolumeFlux<PHYS_ADVECT, T> {
    static constexpr int NV = 1;
    __device__ static void eval(const T* q, T ax, T ay, T, T rx, T ry, T sx, T sy, T* fr, T* fs) {
        const T F = ax * q[0], G = ay * q[0];
        fr[0] = rx * F + ry * G;
        fs[0] = sx * F + sy * G;
    }
};

// dgEulerFoam.C:81-90: gther_U = rhoU / rho, gther_p = (gamma-1)(E - rho |U|^2 / 2); volume
// terms div(U rho), div(U rhoU) + grad(p), div(U E) + div(U p).  Formed directly in the reference directions:
// with the contravariant momenta m_r = rx rhou + ry rhov, m_s = sx rhou + sy rhov and U_r = m_r / rho,
//   rx F + ry G = (m_r, rhou U_r + p rx, rhov U_r + p ry, (E + p) U_r),  likewise for s,
// the same values as rx F + ry G of the Cartesian fluxes in about half the operations.
template <typename T>
struct VolumeFlux<PHYS_EULER, T> {
    static constexpr int NV = 4;
    __device__ static void eval(const T* q, T, T, T gamma, T rx, T ry, T sx, T sy, T* fr, T* fs) {
        const T ru = q[1], rv = q[2], E = q[3];
        const T irho = inv(q[0]);
        const T p = (gamma - T(1)) * (E - T(0.5) * ((ru * ru + rv * rv) * irho));
        const T mr = rx * ru + ry * rv, ms = sx * ru + sy * rv;
        const T Ur = mr * irho, Us = ms * irho, Ep = E + p;
        fr[0] = mr;
        fr[1] = ru * Ur + p * rx;
        fr[2] = rv * Ur + p * ry;
        fr[3] = Ep * Ur;
        fs[0] = ms;
        fs[1] = ru * Us + p * sx;
        fs[2] = rv * Us + p * sy;
        fs[3] = Ep * Us;
    }
};

// Roe flux in the face-normal frame without entropy fix (RoeFlux.C:109-181); M = own side, P = other.
template <typename T>
__device__ __forceinline__ void roe_flux(T g, T nx, T ny, const T* M, const T* P, T* F) {
    const T QP2 = nx * P[1] + ny * P[2], QM2 = nx * M[1] + ny * M[2];
    const T QP3 = nx * P[2] - ny * P[1], QM3 = nx * M[2] - ny * M[1];
    const T rhoP = P[0], rhoM = M[0];
    const T uM = QM2 / rhoM, uP = QP2 / rhoP, vM = QM3 / rhoM, vP = QP3 / rhoP;
    const T pM = (g - T(1)) * (M[3] - T(0.5) * (QM2 * uM + QM3 * vM));
    const T pP = (g - T(1)) * (P[3] - T(0.5) * (QP2 * uP + QP3 * vP));
    const T HM = (M[3] + pM) / rhoM, HP = (P[3] + pP) / rhoP;
    T fr = (QM2 + QP2) / T(2);
    T fu = (QM2 * uM + pM + QP2 * uP + pP) / T(2);
    T fv = (QM3 * uM + QP3 * uP) / T(2);
    T fe = (uM * (M[3] + pM) + uP * (P[3] + pP)) / T(2);
    const T rMs = sqrt(rhoM), rPs = sqrt(rhoP);
    const T rhob = rMs * rPs;
    const T u = (rMs * uM + rPs * uP) / (rMs + rPs);
    const T v = (rMs * vM + rPs * vP) / (rMs + rPs);
    const T H = (rMs * HM + rPs * HP) / (rMs + rPs);
    const T c2 = (g - T(1)) * (H - T(0.5) * (u * u + v * v));
    const T c = sqrt(fabs(c2));
    const T dw1 = (T(-0.5) * rhob * (uP - uM) / c + T(0.5) * (pP - pM) / c2) * fabs(u - c);
    const T dw2 = ((rhoP - rhoM) - (pP - pM) / c2) * fabs(u);
    const T dw3 = (rhob * (vP - vM)) * fabs(u);
    const T dw4 = (T(0.5) * rhob * (uP - uM) / c + T(0.5) * (pP - pM) / c2) * fabs(u + c);
    fr -= (dw1 + dw2 + dw4) / T(2);
    fu -= (dw1 * (u - c) + dw2 * u + dw4 * (u + c)) / T(2);
    fv -= (dw1 * v + dw2 * v + dw3 + dw4 * v) / T(2);
    fe -= (dw1 * (H - u * c) + dw2 * (u * u + v * v) / T(2) + dw3 * v + dw4 * (H + u * c)) / T(2);
    F[0] = fr;
    F[1] = nx * fu - ny * fv;
    F[2] = ny * fu + nx * fv;
    F[3] = fe;
}

// The seed of quotient(): one Newton step, good to some 2^-48.
__device__ __forceinline__ double inv_seed(double x) {
    const double r = __builtin_amdgcn_rcp(x);
    return fma(fma(-x, r, 1.0), r, r);
}
// a / b from r close to 1 / b: the product's remainder added once more, as a division rounds it but for rare cases
__device__ __forceinline__ double quotient(double a, double b, double r) {
    const double q = a * r;
    return fma(fma(-b, q, a), r, q);
}

// The same in FP64 with every quotient from one of four reciprocals: 16 IEEE divisions and 3 square roots were two thirds
// of the face work.  The remainders count: with bare products a * (1 / b) the flux's rms error was 3 to 6 % above that of
// IEEE quotients (1.49e-16 against 1.44e-16 of the sides' fluxes for subsonic jumps); with them it is the same within
// sampling (tests/abi/roe_accuracy.cpp).  They cost 0.6 us of 44 at order 2, 0.3 of 98 at order 4 (K = 131072) and
// nothing on smaller meshes.
template <>
__device__ __forceinline__ void roe_flux<double>(double g, double nx, double ny, const double* M, const double* P,
                                                 double* F) {
    const double QP2 = nx * P[1] + ny * P[2], QM2 = nx * M[1] + ny * M[2];
    const double QP3 = nx * P[2] - ny * P[1], QM3 = nx * M[2] - ny * M[1];
    const double rhoP = P[0], rhoM = M[0], iM = inv_seed(rhoM), iP = inv_seed(rhoP);
    const double uM = quotient(QM2, rhoM, iM), uP = quotient(QP2, rhoP, iP);
    const double vM = quotient(QM3, rhoM, iM), vP = quotient(QP3, rhoP, iP);
    const double pM = (g - 1.0) * (M[3] - 0.5 * (QM2 * uM + QM3 * vM));
    const double pP = (g - 1.0) * (P[3] - 0.5 * (QP2 * uP + QP3 * vP));
    const double eM = M[3] + pM, eP = P[3] + pP;
    const double rMs = fsqrt(rhoM), rPs = fsqrt(rhoP), rs = rMs + rPs, w = inv_seed(rs), rhob = rMs * rPs;
    const double u = quotient(rMs * uM + rPs * uP, rs, w), v = quotient(rMs * vM + rPs * vP, rs, w);
    const double H = quotient(rMs * quotient(eM, rhoM, iM) + rPs * quotient(eP, rhoP, iP), rs, w);
    const double q2 = 0.5 * (u * u + v * v), c2 = (g - 1.0) * (H - q2);
    const double c = fsqrt(fabs(c2)), ic = inv_seed(c), au = fabs(u);
    const double dp = quotient(pP - pM, c2, copysign(ic * ic, c2)), du = quotient(rhob * (uP - uM), c, ic);
    const double dw1 = 0.5 * (dp - du) * fabs(u - c), dw2 = ((rhoP - rhoM) - dp) * au;
    const double dw3 = rhob * (vP - vM) * au, dw4 = 0.5 * (dp + du) * fabs(u + c);
    const double s = dw1 + dw2 + dw4, uc = u * c;
    const double fr = 0.5 * (QM2 + QP2 - s);
    const double fu = 0.5 * (QM2 * uM + pM + QP2 * uP + pP - (u * s + c * (dw4 - dw1)));
    const double fv = 0.5 * (QM3 * uM + QP3 * uP - (v * s + dw3));
    const double fe = 0.5 * (uM * eM + uP * eP - (dw1 * (H - uc) + dw2 * q2 + dw3 * v + dw4 * (H + uc)));
    F[0] = fr;
    F[1] = nx * fu - ny * fv;
    F[2] = ny * fu + nx * fv;
    F[3] = fe;
}

// local Lax-Friedrichs (Rusanov) flux with pointwise |u.n| + c
template <typename T>
__device__ __forceinline__ void llf_flux(T g, T nx, T ny, const T* M, const T* P, T* F) {
    const T iM = inv(M[0]), iP = inv(P[0]);
    const T uM = M[1] * iM, vM = M[2] * iM, uP = P[1] * iP, vP = P[2] * iP;
    const T pM = (g - T(1)) * (M[3] - T(0.5) * M[0] * (uM * uM + vM * vM));
    const T pP = (g - T(1)) * (P[3] - T(0.5) * P[0] * (uP * uP + vP * vP));
    const T unM = uM * nx + vM * ny, unP = uP * nx + vP * ny;
    const T lM = fabs(unM) + fsqrt(fabs(g * pM * iM)), lP = fabs(unP) + fsqrt(fabs(g * pP * iP));
    const T lam = lM > lP ? lM : lP;
    const T FM[4] = {M[0] * unM, M[1] * unM + pM * nx, M[2] * unM + pM * ny, (M[3] + pM) * unM};
    const T FP[4] = {P[0] * unP, P[1] * unP + pP * nx, P[2] * unP + pP * ny, (P[3] + pP) * unP};
#pragma unroll
    for (int v = 0; v < 4; ++v) F[v] = T(0.5) * (FM[v] + FP[v]) + T(0.5) * lam * (M[v] - P[v]);
}

// ---------------------------------------------------------------- stage kernel
// A value at a wavefront-uniform base plus an unsigned byte offset of the lane: one scalar base and one 32-bit register,
// where a signed element index makes the compiler keep a 64-bit address per access.
__device__ __forceinline__ double at_lane(const double* base, unsigned off) {
    return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(base) + off);
}
__device__ __forceinline__ void put_lane(double* base, unsigned off, double x) {
    *reinterpret_cast<double*>(reinterpret_cast<char*>(base) + off) = x;
}

// Orders a wave's LDS writes before its later LDS reads by other lanes of the same wave.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Other side's face nodes of variable rg for face f of element e (connectivity c): neighbour nodes in reversed
// order, or fixedValue ghost nodes.  The Nfp loads are issued with no branch around them: a face without such
// data (its flux copies the own trace) reads a valid address of its own element, and the caller drops the values
// (the return value says whether they are used), so the loads of several faces can be in flight together.
template <int N, int NV, typename OT>
__device__ __forceinline__ bool gather_face(const StageArgs& a, int c, int f, int e, int rg, OT (&o)[N + 1]) {
    constexpr int Np = (N + 1) * (N + 2) / 2, Nfp = N + 1;
    constexpr size_t GS = size_t(NV) * Np * 16;
    const int v = rg < NV ? rg : 0;
    const bool nb = c >= 0;
    const bool fx = !nb && -c - 1 == BC_FIXED && a.bcq != nullptr;
    const int en = nb ? c >> 2 : e, fn = nb ? c & 3 : 0;
    const double* qn = a.q_in + size_t(en >> 4) * GS + size_t(v) * Np * 16 + (en & 15);
    const double* bq = fx ? a.bcq + ((size_t(v) * a.K + e) * 3 + f) * Nfp : qn;
#pragma unroll
    for (int k = 0; k < Nfp; ++k) {
        const int node = fn == 0 ? face_node<N>(0, N - k) : (fn == 1 ? face_node<N>(1, N - k) : face_node<N>(2, N - k));
        const double* src = fx ? bq + k : qn + node * 16;   // one load from the selected address
        o[k] = OT(*src);
    }
    return nb || fx;
}

}  // namespace dg
