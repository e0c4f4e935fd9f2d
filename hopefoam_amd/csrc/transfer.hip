// Reordering of nodal arrays between the host's element-major order and the device's groups of 16 elements.
//
// One wavefront moves one tile (16 elements x Np nodes of one variable): both sides of a tile are contiguous, the
// transpose goes through LDS with an odd row stride.  The host side is pinned memory that the kernel reads or writes
// across PCIe itself (512 contiguous bytes per instruction), so that the reordering, the padding and the copy are one
// pass; PCIe bounds it (57 GB/s each way).  Before, the host reordered element by element in one thread: a field of
// 117 MB took 46 ms to download.
#include <hip/hip_runtime.h>

#include "dg_common.hpp"
#include "transfer.hpp"

namespace dg {

constexpr int kTileMax = 16 * 45;      // order 8
constexpr int kTileLoads = (kTileMax + 63) / 64;   // of one lane
constexpr int kTileStride = 16 * 45 + 16;   // LDS of one wavefront's tile: 16 rows of an odd stride up to 46

template <bool UNPACK>
__global__ __launch_bounds__(256) void tiles_kernel(NodalArray a, int t0, int t1, double* __restrict__ host) {
    __shared__ double tile[4][kTileStride];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int G = a.tiles_per_var(), P = a.Np | 1, n = 16 * a.Np;
    const size_t h0 = a.host_at(t0);
    double* buf = tile[wave];
    for (int t = t0 + blockIdx.x * 4 + wave; t < t1; t += gridDim.x * 4) {
        const int v = t / G, g = t - v * G;
        const int live = a.K - 16 * g < 16 ? a.K - 16 * g : 16;
        double* h = host + (a.host_at(t) - h0);
        double* d = a.dev + (size_t(g) * a.nvar + v) * n;
        // the whole tile is requested before any of it is put down: a load across PCIe takes longer than the rest
        const int count = UNPACK ? live * a.Np : n;
        const double* src = UNPACK ? h : d;
        double x[kTileLoads];
#pragma unroll
        for (int k = 0; k < kTileLoads; ++k) x[k] = lane + 64 * k < count ? src[lane + 64 * k] : 0.0;
#pragma unroll
        for (int k = 0; k < kTileLoads; ++k) {
            const int i = lane + 64 * k, e = UNPACK ? i / a.Np : i & 15;
            if (i < count) buf[e * P + (UNPACK ? i - e * a.Np : i >> 4)] = x[k];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (UNPACK) {
            for (int i = lane; i < n; i += 64) {
                const int e = i & 15;
                d[i] = buf[(e < live ? e : live - 1) * P + (i >> 4)];
            }
            if (g == G - 1)   // whole groups of padding repeat element K - 1
                for (int gp = G; gp < a.groups; ++gp)
                    for (int i = lane; i < n; i += 64)
                        a.dev[(size_t(gp) * a.nvar + v) * n + i] = buf[(live - 1) * P + (i >> 4)];
        } else {
            for (int i = lane; i < live * a.Np; i += 64) {
                const int e = i / a.Np;
                h[i] = buf[e * P + i - e * a.Np];
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

template <bool UNPACK>
static hipError_t launch_tiles(const NodalArray& a, int t0, int t1, double* host, hipStream_t s) {
    if (16 * a.Np > kTileMax || t1 <= t0) return hipErrorInvalidValue;
    const int blocks = (t1 - t0 + 3) / 4;
    hipLaunchKernelGGL((tiles_kernel<UNPACK>), dim3(blocks < 1024 ? blocks : 1024), dim3(256), 0, s, a, t0, t1, host);
    return hipGetLastError();
}

hipError_t launch_unpack_tiles(const NodalArray& a, int t0, int t1, const double* host, hipStream_t s) {
    return launch_tiles<true>(a, t0, t1, const_cast<double*>(host), s);
}
hipError_t launch_pack_tiles(const NodalArray& a, int t0, int t1, double* host, hipStream_t s) {
    return launch_tiles<false>(a, t0, t1, host, s);
}

}  // namespace dg
