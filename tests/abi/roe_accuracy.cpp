// Rounding of the FP64 Roe flux of the stage kernels (stage_device.hpp), compiled for the host with the hardware's
// reciprocal and reciprocal root modelled to 24 bits: its rms error against extended precision over three kinds of states,
// and that of the same flux with IEEE quotients and roots.  Prints one line per kind: kernel's error, quotients' error.
#include <cmath>
#include <cstdio>
#include <random>

static double bits24(double x) {
    int e;
    const double m = std::frexp(x, &e);
    return std::ldexp(std::nearbyint(m * 16777216.0) / 16777216.0, e);
}
#define __builtin_amdgcn_rcp(x) bits24(1.0 / (x))
#define __builtin_amdgcn_rsq(x) bits24(1.0 / std::sqrt(x))
#define __builtin_amdgcn_class(x, mask) ((x) == 0.0 || (x) == __builtin_huge_val())
#define __builtin_amdgcn_rcpf(x) (1.0f / (x))
#define __builtin_amdgcn_sqrtf(x) std::sqrt(x)
#define __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, x, y, z) (c)
#define __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, x, y, z) (c)
#define __builtin_amdgcn_fence(order, scope)
#define __builtin_amdgcn_wave_barrier()

struct Quot {   // double arithmetic under another name: the flux with quotients
    double v;
    Quot(double x = 0) : v(x) {}
    friend Quot operator+(Quot a, Quot b) { return a.v + b.v; }
    friend Quot operator-(Quot a, Quot b) { return a.v - b.v; }
    friend Quot operator*(Quot a, Quot b) { return a.v * b.v; }
    friend Quot operator/(Quot a, Quot b) { return a.v / b.v; }
    Quot& operator-=(Quot b) { return *this = *this - b; }
    friend Quot sqrt(Quot a) { return std::sqrt(a.v); }
    friend Quot fabs(Quot a) { return std::fabs(a.v); }
};
using std::fabs;
using std::fma;
using std::fmax;
using std::sqrt;

#include "stage_device.hpp"

template <typename T>
static void flux(double nx, double ny, const double* M, const double* P, T* F) {
    T m[4], p[4];
    for (int v = 0; v < 4; ++v) {
        m[v] = T(M[v]);
        p[v] = T(P[v]);
    }
    dg::roe_flux<T>(T(1.4), T(nx), T(ny), m, p, F);
}

int main() {
    for (int kind = 0; kind < 3; ++kind) {
        std::mt19937_64 gen(11 + kind);
        std::uniform_real_distribution<double> U(0, 1);
        auto state = [&](double* q, double rho, double u, double v, double p) {
            q[0] = rho;
            q[1] = rho * u;
            q[2] = rho * v;
            q[3] = p / 0.4 + 0.5 * rho * (u * u + v * v);
        };
        long double ek = 0, eq = 0;
        for (int i = 0; i < 400000; ++i) {
            double M[4], P[4], K[4];
            if (kind == 2) {   // the two sides of a resolved flow
                const double rho = 0.5 + U(gen), u = 1 + 0.5 * (U(gen) - 0.5), v = 0.5 * (U(gen) - 0.5), p = 0.5 + U(gen);
                for (double* q : {M, P})
                    state(q, rho * (1 + 1e-3 * U(gen)), u + 1e-3 * U(gen), v + 1e-3 * U(gen), p * (1 + 1e-3 * U(gen)));
            } else {           // jumps: subsonic, and of every speed
                for (double* q : {M, P}) {
                    if (kind == 0) state(q, 0.5 + U(gen), 1 + 0.5 * (U(gen) - 0.5), 0.5 * (U(gen) - 0.5), 0.5 + U(gen));
                    else state(q, 0.1 + 3 * U(gen), 4 * (U(gen) - 0.5), 4 * (U(gen) - 0.5), 0.1 + 5 * U(gen));
                }
            }
            const double th = 6.283185307179586 * U(gen), nx = std::cos(th), ny = std::sin(th);
            Quot Q[4];
            long double R[4], RM[4], RP[4], n2 = 0, k2 = 0, q2 = 0;
            flux<double>(nx, ny, M, P, K);
            flux<Quot>(nx, ny, M, P, Q);
            flux<long double>(nx, ny, M, P, R);
            flux<long double>(nx, ny, M, M, RM);   // the physical fluxes of the two sides: the size of what is rounded
            flux<long double>(nx, ny, P, P, RP);
            for (int v = 0; v < 4; ++v) {
                n2 += 0.5L * (RM[v] * RM[v] + RP[v] * RP[v]);
                k2 += (K[v] - R[v]) * (K[v] - R[v]);
                q2 += (Q[v].v - R[v]) * (Q[v].v - R[v]);
            }
            ek += k2 / n2;
            eq += q2 / n2;
        }
        std::printf("%.6e %.6e\n", double(std::sqrt(ek / 400000)), double(std::sqrt(eq / 400000)));
    }
}
