// Host side of the field transfers (transfer.hpp): pinned staging in chunks, several workers.
//
// A transfer is cut into chunks of one staging slot.  Each worker takes every workers-th chunk and alternates between
// its two slots: while the device packs (or unpacks) one, the worker copies the other from (or to) the caller's memory.
// One worker copies about 30 GB/s; the first touch of a fresh result array costs as much again; the workers share both.
// Small transfers stay on the calling thread.  Measured, up / down: 117 MB 38.8 / 45.7 ms -> 2.9 / 3.3 ms, 42 MB 15.5 /
// 19.8 -> 1.1 / 1.5 ms, 4.2 MB 306 / 825 -> 145 / 155 us, 0.8 MB 62 / 69 -> 42 / 50 us, 0.3 MB 30 / 32 -> 24 / 27 us.
// Pageable copies of 1 to 80 KB took 12 to 30 us, by where the caller's memory lies, these take 15 to 17; upload, right-hand
// side and download in a row 47 -> 38 us at 40 KB, 61 -> 47 at 16 KB.
#include "transfer.hpp"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <thread>
#include <vector>

#include "dg_common.hpp"

namespace dg {

// Data that pays for one more worker (a thread costs some tens of microseconds to start: with a worker per 2 MiB a field
// of 4 MB took 210 us up, with one 146), and the smallest chunks worth a launch of their own (0.3 MB in two chunks 30 / 28 us,
// in one 24 / 26; smaller down, where the first touch of the caller's memory may overlap with the next chunk's copy).
static constexpr size_t kWorkerBytes = size_t(8) << 20;
static constexpr size_t kChunkUp = size_t(512) << 10, kChunkDown = size_t(384) << 10;

bool Staging::ready(int n) {
    if (slots >= n) return true;
    if (failed) return false;
    double* m = nullptr;
    failed = hipHostMalloc(reinterpret_cast<void**>(&m), size_t(n) * kSlotBytes, hipHostMallocCoherent) != hipSuccess;
    for (int i = 0; i < n && !failed; ++i)
        if (!ev[i]) failed = hipEventCreateWithFlags(&ev[i], hipEventDisableTiming) != hipSuccess;
    if (failed) {
        (void)hipGetLastError();
        if (m) (void)hipHostFree(m);
        return false;
    }
    if (mem) (void)hipHostFree(mem);   // of fewer slots; no transfer is under way
    mem = m;
    slots = n;
    return true;
}

void Staging::release() {
    for (hipEvent_t& e : ev) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
    if (mem) (void)hipHostFree(mem);
    mem = nullptr;
    slots = 0;
}

// without pinned memory: one pageable copy of the whole array, reordered by the host
static hipError_t transfer_pageable(hipStream_t s, const NodalArray& a, double* host, bool to_device) {
    const size_t n = size_t(a.nvar) * a.groups * 16 * a.Np;
    std::vector<double> dev(n);
    hipError_t err;
    if (to_device) {
        for (int v = 0; v < a.nvar; ++v)
            for (int e = 0; e < a.groups * 16; ++e) {
                const double* src = host + (size_t(v) * a.K + std::min(e, a.K - 1)) * a.Np;
                for (int j = 0; j < a.Np; ++j) dev[dev_index(e, v, j, a.nvar, a.Np)] = src[j];
            }
        err = hipMemcpyAsync(a.dev, dev.data(), n * sizeof(double), hipMemcpyHostToDevice, s);
        const hipError_t done = hipStreamSynchronize(s);
        return err != hipSuccess ? err : done;
    }
    if ((err = hipMemcpyAsync(dev.data(), a.dev, n * sizeof(double), hipMemcpyDeviceToHost, s)) != hipSuccess) return err;
    if ((err = hipStreamSynchronize(s)) != hipSuccess) return err;
    for (int v = 0; v < a.nvar; ++v)
        for (int e = 0; e < a.K; ++e)
            for (int j = 0; j < a.Np; ++j)
                host[(size_t(v) * a.K + e) * a.Np + j] = dev[dev_index(e, v, j, a.nvar, a.Np)];
    return hipSuccess;
}

hipError_t transfer_array(int device, hipStream_t s, Staging& st, const NodalArray& a, double* host, bool to_device) {
    std::lock_guard<std::mutex> lock(st.mu);
    const int tiles = a.nvar * a.tiles_per_var();
    const size_t bytes = size_t(a.nvar) * a.K * a.Np * sizeof(double);
    // chunks: whole tiles, at most one slot; workers: one per kWorkerBytes, at most one per two slots
    int workers = int(std::min<size_t>(Staging::kSlots / 2, bytes / kWorkerBytes));
    if (workers < 1) workers = 1;
    const int most = int(Staging::kSlotBytes / (size_t(16) * a.Np * sizeof(double)));
    // (a transfer of a few slots is cut finer, so that the copies and the device's work overlap)
    const int per = std::max(1, std::min(most, (tiles + 4 * workers - 1) / (4 * workers)));
    const int least = std::max(per, std::min(most, int((to_device ? kChunkUp : kChunkDown) / (size_t(16) * a.Np * sizeof(double)))));
    int chunks = (tiles + least - 1) / least;
    // Equal chunks, but for the larger uploads: there what is left over makes a short last chunk, and so a short launch after
    // the host's last copy (4.2 MB up 146 us in equal chunks, 142 so, 6.7 MB 212 and 204; down 150 and 154, 219 and 224)
    const int step = to_device && least == per ? least : (tiles + chunks - 1) / chunks;
    chunks = (tiles + step - 1) / step;
    workers = std::min(workers, chunks);
    if (!st.ready(2 * workers)) return transfer_pageable(s, a, host, to_device);
    // One chunk: nothing to overlap.  (Waiting for the kernel's own completion signal, an event handed to its launch, is 2.5 us
    // shorter, but the next synchronisation of the stream then takes 8: upload, right-hand side, download of 16 KB 47 -> 44
    // us, time loop and download 120 -> 122, upload and synchronise 16.6 -> 22.6.)
    if (chunks == 1) {
        if (to_device) std::memcpy(st.slot(0), host, bytes);
        const hipError_t err = to_device ? launch_unpack_tiles(a, 0, tiles, st.slot(0), s)
                                         : launch_pack_tiles(a, 0, tiles, st.slot(0), s);
        const hipError_t done = hipStreamSynchronize(s);
        if (err != hipSuccess || done != hipSuccess) return err != hipSuccess ? err : done;
        if (!to_device) std::memcpy(host, st.slot(0), bytes);
        return hipSuccess;
    }
    std::atomic<int> failed{int(hipSuccess)};
    auto work = [&](int w) {
        if (w > 0 && hipSetDevice(device) != hipSuccess) {
            failed = int(hipErrorInvalidDevice);
            return;
        }
        int pending[2] = {-1, -1};   // chunk in each of the worker's slots
        auto range = [&](int c, int& t0, int& t1, double*& h, size_t& nb) {
            t0 = c * step;
            t1 = std::min(tiles, t0 + step);
            const size_t b = a.host_at(t0), e = t1 == tiles ? size_t(a.nvar) * a.K * a.Np : a.host_at(t1);
            h = host + b;
            nb = (e - b) * sizeof(double);
        };
        auto check = [&](hipError_t e) {
            if (e != hipSuccess) failed = int(e);
            return e == hipSuccess;
        };
        int t0, t1, k = 0;
        double* h;
        size_t nb;
        auto finish = [&](int i) {   // download: wait for slot i's chunk and hand it over
            if (pending[i] < 0) return true;
            if (!check(hipEventSynchronize(st.ev[2 * w + i]))) return false;
            if (!to_device) {
                range(pending[i], t0, t1, h, nb);
                std::memcpy(h, st.slot(2 * w + i), nb);
            }
            pending[i] = -1;
            return true;
        };
        for (int c = w; c < chunks; c += workers, k ^= 1) {
            if (failed != int(hipSuccess) || !finish(k)) break;
            range(c, t0, t1, h, nb);
            double* slot = st.slot(2 * w + k);
            if (to_device) std::memcpy(slot, h, nb);
            if (!check(to_device ? launch_unpack_tiles(a, t0, t1, slot, s) : launch_pack_tiles(a, t0, t1, slot, s)) ||
                !check(hipEventRecord(st.ev[2 * w + k], s)))
                break;
            pending[k] = c;
        }
        // the slots are free, and the caller's memory done with, when this returns
        const bool first = finish(k), second = finish(k ^ 1);
        (void)first;
        (void)second;
    };
    std::vector<std::thread> pool;
    int started = 1;
    try {
        pool.reserve(size_t(workers));
        for (; started < workers; ++started) pool.emplace_back(work, started);
    } catch (...) {   // no memory or no more threads: their chunks are done below
    }
    work(0);
    for (int w = started; w < workers; ++w) work(w);
    for (std::thread& t : pool) t.join();
    if (failed != int(hipSuccess)) {
        (void)hipStreamSynchronize(s);   // nothing still reads or writes the slots
        return hipError_t(failed.load());
    }
    return hipSuccess;
}

hipError_t fetch_small(hipStream_t s, Staging& st, void* host, const void* dev, size_t bytes, void* host2,
                       const void* dev2, size_t bytes2) {
    std::lock_guard<std::mutex> lock(st.mu);
    const size_t at2 = (bytes + 63) / 64 * 64;
    const bool pinned = st.mem && at2 + bytes2 <= size_t(st.slots) * Staging::kSlotBytes;
    void *a = pinned ? st.slot(0) : host, *b = pinned ? reinterpret_cast<char*>(st.slot(0)) + at2 : host2;
    hipError_t err = hipSuccess;
    if (dev) err = hipMemcpyAsync(a, dev, bytes, hipMemcpyDeviceToHost, s);
    if (dev2 && err == hipSuccess) err = hipMemcpyAsync(b, dev2, bytes2, hipMemcpyDeviceToHost, s);
    const hipError_t done = hipStreamSynchronize(s);
    if (err != hipSuccess || done != hipSuccess) return err != hipSuccess ? err : done;
    if (pinned) {
        if (dev) std::memcpy(host, a, bytes);
        if (dev2) std::memcpy(host2, b, bytes2);
    }
    return hipSuccess;
}

}  // namespace dg
