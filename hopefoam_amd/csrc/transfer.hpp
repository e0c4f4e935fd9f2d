// Nodal arrays between host memory ([var][K][Np]) and the device field layout (dev_index, dg_common.hpp).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <mutex>

namespace dg {

// One array: nvar variables of K elements with Np nodes at dev, padded to groups * 16 elements (padding elements repeat
// element K - 1; the layout keeps a tile of 16 elements x Np nodes per (group, variable)).
struct NodalArray {
    double* dev = nullptr;
    int nvar = 1, K = 0, Np = 0, groups = 0;
    __host__ __device__ int tiles_per_var() const { return (K + 15) / 16; }   // tiles that hold elements
    // first host value of tile t = variable * tiles_per_var + group; consecutive tiles are consecutive in host memory
    __host__ __device__ size_t host_at(int t) const {
        const int G = tiles_per_var();
        return (size_t(t / G) * K + size_t(t % G) * 16) * Np;
    }
};

// Pinned staging memory of a context, allocated with the first transfer that needs it and freed with the context: two slots
// per worker, so that the copy of one overlaps the device's work on the other, at most kSlots.
struct Staging {
    static constexpr int kSlots = 16;
    static constexpr size_t kSlotBytes = size_t(1) << 20;   // 16 MiB with every slot
    std::mutex mu;                 // one transfer at a time
    double* mem = nullptr;
    int slots = 0;                 // of mem
    hipEvent_t ev[kSlots] = {};
    bool failed = false;           // no (more) pinned memory: transfers go through pageable copies
    bool ready(int n);             // n slots and their events are there
    void release();
    double* slot(int i) const { return mem + size_t(i) * (kSlotBytes / sizeof(double)); }
};

// tiles [t0, t1) of a from / to the packed host order at host (device-accessible memory)
hipError_t launch_unpack_tiles(const NodalArray& a, int t0, int t1, const double* host, hipStream_t s);
hipError_t launch_pack_tiles(const NodalArray& a, int t0, int t1, double* host, hipStream_t s);

// the whole array from / to host memory, ordered behind the work on stream s and complete on return
hipError_t transfer_array(int device, hipStream_t s, Staging& st, const NodalArray& a, double* host, bool to_device);

// Small results to host memory, behind the work on s; complete on return.  Two pieces (either dev may be null) share
// one synchronisation, through the staging slots where they fit and the context has them already (nothing is allocated).
hipError_t fetch_small(hipStream_t s, Staging& st, void* host, const void* dev, size_t bytes, void* host2,
                       const void* dev2, size_t bytes2);

}  // namespace dg
