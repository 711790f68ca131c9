// vrn_xfer.hip -- see vrn_xfer.hpp.
#include "vrn_xfer.hpp"

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>

namespace {

// Measured on a 384^3 state (2.37 GB), to / from the device: runtime 27 / 17
// GB/s (into pages not yet touched 10), this 54 / 48 (39).  4 threads and 2
// slots each keep the link busy (6 and 8 threads, 4 slots: the same); a copy
// of 1 or 2 MB on one stream leaves it idle for 15 us (31 or 40 GB/s), which
// a second stream and 4 MB cover.
constexpr int THREADS = 4;  // copying threads, the caller among them
constexpr int SLOTS = 2;    // of each thread: one being copied, one on the link
constexpr int STREAMS = 2;
constexpr size_t SLOT = (size_t)4 << 20, SLICE_MIN = (size_t)1 << 20;
// From LARGE_UP and LARGE_DOWN on, staging pays for starting the threads
// (14 MB: 0.56 against 0.41 ms up, 0.48 against 0.83 ms down); its memory and
// streams cost 3 to 5 ms once, so the first WORTH bytes of large copies go
// without.
constexpr size_t LARGE_UP = (size_t)24 << 20, LARGE_DOWN = (size_t)8 << 20, WORTH = (size_t)64 << 20;

std::mutex g_mutex;  // holds the staging memory: one copy uses it at a time
char *g_stage = nullptr;
hipEvent_t g_event[THREADS * SLOTS] = {};
hipEvent_t g_order = nullptr;    // where the caller's stream stood
hipStream_t g_stream[STREAMS] = {};
int g_event_dev = -1;  // device the events and streams belong to
size_t g_moved = 0;    // bytes of large copies while there was no staging memory
std::atomic<int> g_handles{0};

void drop_queues()
{
    for (hipStream_t &q : g_stream) {
        if (q) (void)hipStreamDestroy(q);
        q = nullptr;
    }
    for (hipEvent_t &e : g_event) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
    if (g_order) (void)hipEventDestroy(g_order);
    g_order = nullptr;
    g_event_dev = -1;
}

// Staging memory, streams and events for the current device; false if there
// are none.
bool ready(int dev)
{
    if (!g_stage &&
        hipHostMalloc(reinterpret_cast<void **>(&g_stage), SLOT * SLOTS * THREADS, hipHostMallocPortable) != hipSuccess) {
        (void)hipGetLastError();
        g_stage = nullptr;
        return false;
    }
    if (g_event_dev == dev) return true;
    drop_queues();
    bool ok = hipEventCreateWithFlags(&g_order, hipEventDisableTiming) == hipSuccess;
    for (hipEvent_t &e : g_event) ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
    for (hipStream_t &q : g_stream) ok = ok && hipStreamCreateWithFlags(&q, hipStreamNonBlocking) == hipSuccess;
    if (!ok) {
        (void)hipGetLastError();
        drop_queues();
        return false;
    }
    g_event_dev = dev;
    return true;
}

// Whether CPU threads may copy at this address: memory that the runtime knows
// (pinned, managed, a device's) is left to it.
bool pageable(const void *host)
{
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, host) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return a.type == hipMemoryTypeUnregistered;
}

// One thread's share of a staged copy: the slices k = t, t + THREADS, ...
// To the device: fill a slot, put it on the stream.  From it: put the next
// slot on the stream, then empty the one before.
hipError_t share(int t, int dev, bool down, char *host, char *device, size_t n, std::atomic<int> &failed)
{
    hipError_t e = hipSetDevice(dev);
    const hipStream_t s = g_stream[t % STREAMS];
    // enough slices that every thread overlaps its copies with the link
    const size_t part = std::min(SLOT, std::max(SLICE_MIN, n / (4 * THREADS)));
    const long slices = (long)((n + part - 1) / part);
    char *slot[SLOTS];
    for (int j = 0; j < SLOTS; j++) slot[j] = g_stage + (size_t)(t * SLOTS + j) * SLOT;
    hipEvent_t *ev = g_event + t * SLOTS;
    auto len = [&](long k) { return std::min(part, n - (size_t)k * part); };
    long used = 0;  // slots put on the stream
    auto finish = [&](long i, long k) {
        // slice k went into slot i % SLOTS
        hipError_t w = hipEventSynchronize(ev[i % SLOTS]);
        if (w == hipSuccess && down && e == hipSuccess)
            std::memcpy(host + (size_t)k * part, slot[i % SLOTS], len(k));
        if (e == hipSuccess) e = w;
    };
    for (long k = t; k < slices && e == hipSuccess && !failed.load(std::memory_order_relaxed); k += THREADS) {
        const int j = (int)(used % SLOTS);
        if (used >= SLOTS) finish(used - SLOTS, k - (long)SLOTS * THREADS);
        if (e != hipSuccess) break;
        const size_t at = (size_t)k * part;
        if (down) {
            e = hipMemcpyAsync(slot[j], device + at, len(k), hipMemcpyDeviceToHost, s);
        } else {
            std::memcpy(slot[j], host + at, len(k));
            e = hipMemcpyAsync(device + at, slot[j], len(k), hipMemcpyHostToDevice, s);
        }
        if (e == hipSuccess) e = hipEventRecord(ev[j], s);
        if (e == hipSuccess) used++;
    }
    // the slots still on the stream
    for (long i = std::max(0L, used - SLOTS); i < used; i++) finish(i, t + i * THREADS);
    if (e != hipSuccess) (void)hipStreamSynchronize(s);  // also a copy whose event could not be recorded
    if (e != hipSuccess) failed.store(1, std::memory_order_relaxed);
    return e;
}

// Staged copy; false if it cannot be made this way (nothing was copied).
bool staged(bool down, void *host, void *device, size_t n, hipStream_t s, hipError_t *result)
{
    std::unique_lock<std::mutex> lk(g_mutex, std::try_to_lock);
    if (!lk.owns_lock() || g_handles.load() == 0) return false;
    if (!g_stage && (g_moved += n) < WORTH) return false;
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || !ready(dev)) return false;
    // the copies come after what stream s holds; what is put on s after this
    // call comes after them, since it returns when they are done
    bool ok = hipEventRecord(g_order, s) == hipSuccess;
    for (hipStream_t q : g_stream) ok = ok && hipStreamWaitEvent(q, g_order, 0) == hipSuccess;
    if (!ok) {
        (void)hipGetLastError();
        return false;
    }
    std::atomic<int> failed{0};
    hipError_t e[THREADS] = {};
    std::thread th[THREADS];
    bool run[THREADS] = {};
    for (int t = 1; t < THREADS; t++) {
        try {
            th[t] = std::thread([&, t] {
                e[t] = share(t, dev, down, static_cast<char *>(host), static_cast<char *>(device), n, failed);
            });
            run[t] = true;
        } catch (const std::exception &) {  // no thread or memory to be had: the caller takes its share
        }
    }
    for (int t = 0; t < THREADS; t++)
        if (!run[t])
            e[t] = share(t, dev, down, static_cast<char *>(host), static_cast<char *>(device), n, failed);
    for (int t = 1; t < THREADS; t++)
        if (run[t]) th[t].join();
    *result = hipSuccess;
    for (int t = 0; t < THREADS; t++)
        if (*result == hipSuccess) *result = e[t];
    return true;
}

}  // namespace

namespace vrn_xfer {

void retain() { g_handles++; }

void release()
{
    if (--g_handles > 0) return;
    std::lock_guard<std::mutex> lk(g_mutex);
    if (g_handles.load() > 0) return;
    drop_queues();
    if (g_stage) (void)hipHostFree(g_stage);
    g_stage = nullptr;
    g_moved = 0;
}

hipError_t h2d(void *dev, const void *host, size_t n, hipStream_t s)
{
    hipError_t e;
    if (n >= LARGE_UP && pageable(host) && staged(false, const_cast<void *>(host), dev, n, s, &e)) return e;
    return hipMemcpyAsync(dev, host, n, hipMemcpyHostToDevice, s);
}

hipError_t d2h(void *host, const void *dev, size_t n, hipStream_t s)
{
    hipError_t e;
    if (n >= LARGE_DOWN && pageable(host) && staged(true, host, const_cast<void *>(dev), n, s, &e)) return e;
    e = hipMemcpyAsync(host, dev, n, hipMemcpyDeviceToHost, s);
    return e == hipSuccess ? hipStreamSynchronize(s) : e;
}

}  // namespace vrn_xfer
