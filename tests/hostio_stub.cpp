// Drives the staged host transfers of hostio.hip on the CPU: the HIP calls that it
// makes are host copies here, and an event can be held back.  Prints one line a
// check ("ok" or "FAIL") and returns the number of failures.
#include "../midapack_amd/csrc/mgpu_internal.h"

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <future>
#include <mutex>
#include <numeric>
#include <thread>

namespace {
struct Gate {
    std::mutex mu;
    std::condition_variable cv;
    bool open = true;
    std::atomic<int> waiting{0};
    void set(bool v) {
        std::lock_guard<std::mutex> g(mu);
        open = v;
        cv.notify_all();
    }
    void pass() {
        std::unique_lock<std::mutex> g(mu);
        waiting++;
        cv.wait(g, [&] { return open; });
        waiting--;
    }
};
Gate held_event;  // its address is the event handle
const hipEvent_t kHeld = reinterpret_cast<hipEvent_t>(&held_event);
int dummy;
std::atomic<int> copies{0};           // device copies made
const unsigned char *locked = nullptr;  // the page-locked array
std::atomic<int> last_error{hipSuccess};
hipStream_t last_stream = nullptr;      // of the last queued copy
const hipStream_t kOwn = reinterpret_cast<hipStream_t>(&copies);
}  // namespace

extern "C" {
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stub"; }
hipError_t hipGetLastError() { return (hipError_t) last_error.exchange(hipSuccess); }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
    if (!locked || p != locked) {
        last_error = hipErrorInvalidValue;
        return hipErrorInvalidValue;
    }
    a->type = hipMemoryTypeHost;
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return *p = malloc(n), hipSuccess; }
hipError_t hipHostFree(void *p) { return free(p), hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    return copies++, memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st) {
    if (st == kOwn || !last_stream) last_stream = st;
    return copies++, memcpy(d, s, n), hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    return *s = reinterpret_cast<hipStream_t>(&dummy), hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    return *e = reinterpret_cast<hipEvent_t>(&dummy), hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) {
    if (e == kHeld) held_event.pass();
    return hipSuccess;
}
const char *mappraiser_gpu_last_error() { return ""; }
}
namespace mgpu {
void set_error(const char *, ...) {}
}  // namespace mgpu

using namespace mgpu;
using Bytes = std::vector<unsigned char>;

static int failures = 0;
static void check(bool ok, const char *what, size_t bytes) {
    printf("%s %s, %zu bytes\n", ok ? "ok" : "FAIL", what, bytes);
    fflush(stdout);
    failures += !ok;
}

static Bytes pattern(size_t n) {
    Bytes b(n);
    unsigned v = 12345;
    for (auto &x : b) x = (unsigned char) ((v = v * 1664525u + 1013904223u) >> 24);
    return b;
}

// f on a thread of its own ends within five seconds; the gate opens either way
template <typename F>
static bool ends(Gate &gate, F f) {
    auto fut = std::async(std::launch::async, f);
    const bool in_time = fut.wait_for(std::chrono::seconds(5)) == std::future_status::ready;
    gate.set(true);
    return fut.get() == MGPU_OK && in_time;
}

int main() {
    const size_t MiB = (size_t) 1 << 20;
    // every kind of transfer with the pool free, at the sizes where its form changes
    for (size_t n : {MiB * 0 + 12, MiB / 4 - 12, MiB / 4 + 12, 4 * MiB + 12, 8 * MiB - 12, 8 * MiB, 16 * MiB - 12, 16 * MiB + 12, 100 * MiB + 24}) {
        const Bytes src = pattern(n);
        Bytes dst(n), back(n);
        check(h2d_staged(0, dst.data(), src.data(), n, nullptr) == MGPU_OK && dst == src, "upload", n);
        Bytes made(n);
        const int rc = h2d_staged_fill(0, made.data(), n, [&](size_t off, void *c, size_t len) {
            memcpy(c, src.data() + off, len);
        });
        check(rc == MGPU_OK && made == src, "produced upload", n);
        check(d2h_staged(0, back.data(), src.data(), n, nullptr, nullptr, nullptr) == MGPU_OK && back == src, "download", n);
        Bytes used(n);
        const StageConsumer take = [&](size_t off, const void *c, size_t len) { memcpy(used.data() + off, c, len); };
        check(d2h_staged(0, nullptr, src.data(), n, nullptr, nullptr, &take) == MGPU_OK && used == src, "consumed download", n);
    }
    // one plain copy up to the sizes where staging is the faster form
    for (size_t n : {4 * MiB, 8 * MiB - 8, 8 * MiB, 16 * MiB}) {
        const Bytes src = pattern(n);
        Bytes up(n), down(n);
        copies = 0;
        check(h2d_staged(0, up.data(), src.data(), n, nullptr) == MGPU_OK && (copies == 1) == (n < 8 * MiB), "upload's form", n);
        copies = 0;
        check(d2h_staged(0, down.data(), src.data(), n, nullptr, nullptr, nullptr) == MGPU_OK && (copies == 1) == (n < 8 * MiB),
              "download's form", n);
    }
    // a plain download is queued on the caller's stream and waits for nothing else
    {
        const Bytes src = pattern(MiB);
        Bytes down(MiB);
        last_stream = nullptr;
        held_event.set(false);
        check(ends(held_event, [&] { return d2h_staged(0, down.data(), src.data(), MiB, kHeld, kOwn, nullptr); }) &&
                      last_stream == kOwn && down == src,
              "download queued on its stream", MiB);
    }
    // page-locked arrays are copied directly, and asking about the others leaves no error behind
    check(last_error == hipSuccess, "no error left", 0);
    for (size_t n : {16 * MiB, 64 * MiB + 24}) {
        const Bytes src = pattern(n);
        Bytes up(n), down(n);
        copies = 0;
        locked = src.data();
        check(h2d_staged(0, up.data(), src.data(), n, nullptr) == MGPU_OK && copies == 1 && up == src,
              "page-locked upload", n);
        copies = 0;
        locked = down.data();
        check(d2h_staged(0, down.data(), src.data(), n, nullptr, nullptr, nullptr) == MGPU_OK && copies == 1 && down == src,
              "page-locked download", n);
        locked = nullptr;
    }
    // a transfer that another one holds up goes straight through as a plain copy
    for (size_t n : {MiB, 4 * MiB, 16 * MiB, 64 * MiB}) {
        const Bytes src = pattern(n);
        Bytes up(n), down(n);
        Gate gate;
        auto occupy = [&](std::thread &t) {  // holds the pool until the gate opens
            gate.set(false);
            t = std::thread([&] {
                static unsigned char sink[4096];
                h2d_staged_fill(0, sink, sizeof(sink), [&](size_t, void *, size_t) { gate.pass(); });
            });
            while (!gate.waiting) std::this_thread::yield();
        };
        std::thread a, b;
        occupy(a);
        check(ends(gate, [&] { return h2d_staged(0, up.data(), src.data(), n, nullptr); }) && up == src,
              "upload beside a busy pool", n);
        a.join();
        occupy(b);
        check(ends(gate, [&] { return d2h_staged(0, down.data(), src.data(), n, nullptr, nullptr, nullptr); }) && down == src,
              "download beside a busy pool", n);
        b.join();
        // a download that waits for the device does not hold the pool meanwhile
        Bytes made(n), used(n);
        const StageConsumer take = [&](size_t off, const void *c, size_t len) { memcpy(used.data() + off, c, len); };
        held_event.set(false);
        std::thread w([&] { d2h_staged(0, nullptr, src.data(), n, kHeld, nullptr, &take); });
        while (!held_event.waiting) std::this_thread::yield();
        check(ends(held_event, [&] {
                  return h2d_staged_fill(0, made.data(), n, [&](size_t off, void *c, size_t len) {
                      memcpy(c, src.data() + off, len);
                  });
              }) && made == src, "produced upload beside a download that waits for its event", n);
        w.join();
        check(used == src, "that download", n);
    }
    return failures;
}
