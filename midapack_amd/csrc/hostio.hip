// hostio.hip -- large copies between the caller's (pageable) host arrays and
// the device.
//
// MLmap's arrays (pointing, weights, signal, noise) are ordinary pageable host
// memory; a plain hipMemcpy from pageable memory runs at a fraction of the PCIe
// rate.  Here a pool of pinned staging buffers is shared by a few host worker
// threads: each worker copies its chunks of the caller's array into its own
// pinned buffers (two in flight) and queues the DMA on its own stream, so the
// host copies of one worker overlap the DMA of the others.  The pool is
// allocated once per process (hipHostMalloc; freed by mappraiser_gpu_finalize)
// and used by one transfer at a time: while it is taken, copies of caller's
// arrays go as plain copies beside it and only h2d_staged_fill, which has no other
// form, waits for it.  A staged transfer is complete when the call returns: the
// caller's stream never waits on the pool's events, which the next transfer
// (possibly another host thread's) records again as soon as the pool is released.
#include "mgpu_internal.h"

#include <algorithm>
#include <cstring>
#include <mutex>
#include <thread>

namespace mgpu {

namespace {

constexpr size_t kStageChunk = (size_t) 12 << 20;  // bytes per chunk at most (a whole number of units)
constexpr size_t kStageUnit = 48 << 10;            // chunks are multiples of it, and so of 8, 12 and 16
// Plain copies below kStageMin go through hipMemcpyAsync; copies with host work
// on every chunk (packing, side effects) are shared by a thread per kStageWork
// bytes, two chunks each.  (A drop-in solve of 3.1 M samples, whose 38 MB of local
// indices and side effects one thread took through a plain copy: 27 -> 11 ms.)  The
// threads' start costs more than they save below it: a solve with two uploads from
// arrays that change takes 0.64 ms staged and 0.58 plain with 4.8 MB each, 0.73 and
// 0.71 with 6.4, 0.78 and 0.80 with 8, 0.89 and 1.00 with 10.6, 1.10 and 1.37 with 16
// (from the same arrays every time 0.66 and 0.51, 0.73 and 0.60, 0.79 and 0.68, 0.93
// and 0.84, 1.11 and 1.18); one that downloads a map of 5 MB 1.69 and 1.64, of 8.3 MB
// 2.39 and 2.46, of 13 MB 3.48 and 3.70.
constexpr size_t kStageMin = (size_t) 8 << 20;
constexpr size_t kStageWork = (size_t) 256 << 10;
constexpr int kMaxWorkers = 8;
constexpr int kMaxDevices = 16;

struct StagePool {
    std::mutex busy;       // held for the whole of one staged transfer
    std::mutex init_mu;
    int workers = 0;
    unsigned char *pinned = nullptr;  // workers * 2 * kStageChunk
    hipStream_t ws[kMaxDevices][kMaxWorkers] = {};
    hipEvent_t ev[kMaxDevices][kMaxWorkers][2] = {};
    hipEvent_t done[kMaxDevices][kMaxWorkers] = {};
    bool dev_ready[kMaxDevices] = {};
};

StagePool g_pool;

// workers and chunk size of a transfer
struct StageSplit {
    int workers;
    size_t chunk, n;
    StageSplit(size_t bytes, int most) {
        workers = (int) std::min<size_t>((size_t) most, std::max<size_t>(1, bytes / kStageWork));
        const size_t share = bytes / (2 * (size_t) workers) + 1;
        chunk = std::min(kStageChunk, (share + kStageUnit - 1) / kStageUnit * kStageUnit);
        n = (bytes + chunk - 1) / chunk;
    }
};

unsigned char *buffer(int w, int b) { return g_pool.pinned + ((size_t) w * 2 + b) * kStageChunk; }

// pinned buffers (once per process) and the device's streams and events (once per device)
int pool_ready(int device) {
    std::lock_guard<std::mutex> g(g_pool.init_mu);
    if (!g_pool.pinned) {
        const unsigned hc = std::max(1u, std::thread::hardware_concurrency());
        g_pool.workers = (int) std::min<unsigned>(kMaxWorkers, hc);
        void *p = nullptr;
        MGPU_HIP(hipHostMalloc(&p, (size_t) g_pool.workers * 2 * kStageChunk, hipHostMallocPortable));
        g_pool.pinned = (unsigned char *) p;
    }
    MGPU_ARG(device >= 0 && device < kMaxDevices, "device %d: host staging supports %d devices", device,
             kMaxDevices);
    if (!g_pool.dev_ready[device]) {
        for (int w = 0; w < g_pool.workers; w++) {
            MGPU_HIP(hipStreamCreateWithFlags(&g_pool.ws[device][w], hipStreamNonBlocking));
            for (int b = 0; b < 2; b++)
                MGPU_HIP(hipEventCreateWithFlags(&g_pool.ev[device][w][b], hipEventDisableTiming));
            MGPU_HIP(hipEventCreateWithFlags(&g_pool.done[device][w], hipEventDisableTiming));
        }
        g_pool.dev_ready[device] = true;
    }
    return MGPU_OK;
}

// Arrays that the device reaches by itself (hipHostMalloc, torch's pinned tensors)
// gain nothing from staging: their copies are one DMA at the full PCIe rate (two
// uploads of 16 MB staged 1.23 ms a solve, directly 0.92; of 128 MB 6.3 and 5.3).
bool page_locked(const void *h) {
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, h) != hipSuccess) {
        (void) hipGetLastError();  // memory that HIP does not know: not an error of this call
        return false;
    }
    return a.type == hipMemoryTypeHost;
}

// run fn(w) on `workers` threads (w = 0 on the calling thread); the first
// non-zero status is returned (with its error message)
template <typename F>
int run_workers(int device, int workers, F fn) {
    std::vector<int> rc((size_t) workers, MGPU_OK);
    std::vector<std::string> err((size_t) workers);
    std::vector<std::thread> th;
    for (int w = 1; w < workers; w++)
        th.emplace_back([&, w] {
            if (hipSetDevice(device) != hipSuccess) {
                rc[w] = MGPU_EHIP;
                err[w] = "hipSetDevice failed in a staging thread";
                return;
            }
            rc[w] = fn(w);
            if (rc[w]) err[w] = mappraiser_gpu_last_error();
        });
    rc[0] = fn(0);
    if (rc[0]) err[0] = mappraiser_gpu_last_error();
    for (auto &t : th) t.join();
    for (int w = 0; w < workers; w++)
        if (rc[w]) {
            set_error("%s", err[w].c_str());
            return rc[w];
        }
    return MGPU_OK;
}

}  // namespace

int h2d_staged(int device, void *d, const void *h, size_t bytes, hipStream_t s) {
    std::unique_lock<std::mutex> lk(g_pool.busy, std::defer_lock);
    if (bytes >= kStageMin && !page_locked(h)) lk.try_lock();
    if (!lk.owns_lock()) {  // small, page-locked or pool busy: another thread's transfer may hold it for long
        MGPU_HIP(hipMemcpyAsync(d, h, bytes, hipMemcpyHostToDevice, s));
        return MGPU_OK;
    }
    MGPU_RET(pool_ready(device));
    const StageSplit sp(bytes, g_pool.workers);
    const int W = sp.workers;
    const size_t nch = sp.n;
    unsigned char *dd = (unsigned char *) d;
    const unsigned char *hh = (const unsigned char *) h;
    MGPU_RET(run_workers(device, W, [&](int w) -> int {
        hipStream_t st = g_pool.ws[device][w];
        int j = 0;
        for (size_t k = (size_t) w; k < nch; k += (size_t) W, j++) {
            const int b = j & 1;
            const size_t off = k * sp.chunk, len = std::min(sp.chunk, bytes - off);
            // the buffer's previous DMA (of this or an earlier transfer) has finished
            MGPU_HIP(hipEventSynchronize(g_pool.ev[device][w][b]));
            std::memcpy(buffer(w, b), hh + off, len);
            MGPU_HIP(hipMemcpyAsync(dd + off, buffer(w, b), len, hipMemcpyHostToDevice, st));
            MGPU_HIP(hipEventRecord(g_pool.ev[device][w][b], st));
        }
        MGPU_HIP(hipEventRecord(g_pool.done[device][w], st));
        return MGPU_OK;
    }));
    // complete before the pool is released (and its events recorded again)
    for (int w = 0; w < W; w++) MGPU_HIP(hipEventSynchronize(g_pool.done[device][w]));
    return MGPU_OK;
}

int h2d_staged_fill(int device, void *d, size_t bytes, const StageProducer &fill) {
    std::lock_guard<std::mutex> lk(g_pool.busy);
    MGPU_RET(pool_ready(device));
    const StageSplit sp(bytes, g_pool.workers);
    const int W = sp.workers;
    const size_t nch = sp.n;
    unsigned char *dd = (unsigned char *) d;
    MGPU_RET(run_workers(device, W, [&](int w) -> int {
        hipStream_t st = g_pool.ws[device][w];
        int j = 0;
        for (size_t k = (size_t) w; k < nch; k += (size_t) W, j++) {
            const int b = j & 1;
            const size_t off = k * sp.chunk, len = std::min(sp.chunk, bytes - off);
            MGPU_HIP(hipEventSynchronize(g_pool.ev[device][w][b]));
            fill(off, buffer(w, b), len);
            MGPU_HIP(hipMemcpyAsync(dd + off, buffer(w, b), len, hipMemcpyHostToDevice, st));
            MGPU_HIP(hipEventRecord(g_pool.ev[device][w][b], st));
        }
        MGPU_HIP(hipEventRecord(g_pool.done[device][w], st));
        return MGPU_OK;
    }));
    for (int w = 0; w < W; w++) MGPU_HIP(hipEventSynchronize(g_pool.done[device][w]));
    return MGPU_OK;
}

int d2h_staged(int device, void *h, const void *d, size_t bytes, hipEvent_t after, hipStream_t s,
               const StageConsumer *consume) {
    std::unique_lock<std::mutex> lk(g_pool.busy, std::defer_lock);
    if (consume ? bytes >= kStageWork : bytes >= kStageMin && !page_locked(h)) {
        MGPU_HIP(hipEventSynchronize(after));  // before the pool is taken; its streams wait on no other stream
        lk.try_lock();
    }
    if (!lk.owns_lock()) {
        // small, page-locked or pool busy: one copy, then the consumer over the whole array.
        // (A map queued on the solve's stream: small solves take 10-20 us less than
        // with a wait for the event and a blocking copy.)
        if (consume) {
            MGPU_HIP(hipEventSynchronize(after));
            std::vector<unsigned char> tmp(bytes);
            MGPU_HIP(hipMemcpy(tmp.data(), d, bytes, hipMemcpyDeviceToHost));
            (*consume)(0, tmp.data(), bytes);
        } else {
            MGPU_HIP(hipMemcpyAsync(h, d, bytes, hipMemcpyDeviceToHost, s));
        }
        return MGPU_OK;
    }
    MGPU_RET(pool_ready(device));
    const StageSplit sp(bytes, g_pool.workers);
    const int W = sp.workers;
    const size_t nch = sp.n;
    const unsigned char *dd = (const unsigned char *) d;
    unsigned char *hh = (unsigned char *) h;
    return run_workers(device, W, [&](int w) -> int {
        hipStream_t st = g_pool.ws[device][w];
        auto issue = [&](size_t k, int b) -> int {
            const size_t off = k * sp.chunk, len = std::min(sp.chunk, bytes - off);
            MGPU_HIP(hipEventSynchronize(g_pool.ev[device][w][b]));
            MGPU_HIP(hipMemcpyAsync(buffer(w, b), dd + off, len, hipMemcpyDeviceToHost, st));
            MGPU_HIP(hipEventRecord(g_pool.ev[device][w][b], st));
            return MGPU_OK;
        };
        size_t k = (size_t) w;
        int j = 0;
        if (k < nch) MGPU_RET(issue(k, 0));
        for (; k < nch; k += (size_t) W, j++) {
            const int b = j & 1;
            if (k + W < nch) MGPU_RET(issue(k + W, b ^ 1));  // next chunk in flight meanwhile
            MGPU_HIP(hipEventSynchronize(g_pool.ev[device][w][b]));
            const size_t off = k * sp.chunk, len = std::min(sp.chunk, bytes - off);
            if (consume)
                (*consume)(off, buffer(w, b), len);
            else
                std::memcpy(hh + off, buffer(w, b), len);
        }
        return MGPU_OK;
    });
}

void staging_free() {
    std::lock_guard<std::mutex> b(g_pool.busy);
    std::lock_guard<std::mutex> g(g_pool.init_mu);
    int cur = 0;
    (void) hipGetDevice(&cur);
    for (int dv = 0; dv < kMaxDevices; dv++) {
        if (!g_pool.dev_ready[dv]) continue;
        if (hipSetDevice(dv) != hipSuccess) continue;
        for (int w = 0; w < g_pool.workers; w++) {
            (void) hipStreamSynchronize(g_pool.ws[dv][w]);
            (void) hipStreamDestroy(g_pool.ws[dv][w]);
            for (int b = 0; b < 2; b++) (void) hipEventDestroy(g_pool.ev[dv][w][b]);
            (void) hipEventDestroy(g_pool.done[dv][w]);
        }
        g_pool.dev_ready[dv] = false;
    }
    (void) hipSetDevice(cur);
    if (g_pool.pinned) (void) hipHostFree(g_pool.pinned);
    g_pool.pinned = nullptr;
}

}  // namespace mgpu
