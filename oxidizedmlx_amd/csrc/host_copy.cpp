// host_copy.cpp — copies of large results into the caller's pageable memory
// (Stream::get_buffer, crates/mlx-core/src/backend.rs:162-164, and the
// decoder's logits).
//
// hipMemcpy into pageable memory goes through the runtime's staging with one
// thread, which also takes the page faults of a fresh destination: 17 GB/s on
// memory that is already mapped, about 4 GB/s on new memory, where the link
// carries 55 GB/s into pinned memory. Here several threads each move chunks
// through a pinned slot of their own (host_slots.hpp), so one chunk's copy by
// the CPU (and its page faults) runs beside the others' transfers.
// us through the runtime's way / here with kept slots, into new pages (and
// into mapped ones): 128 KiB 92 / 30 (17 / 16), 1 MiB 290 / 215 (65 / 61), 2 MiB
// 580 / 430 (121 / 113), 4 MiB 1150 / 920 (240 / 203), 16 MiB 4550 / 3600 (950 /
// 580), 64 MiB 18100 / 14200 (3900 / 1820).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <system_error>
#include <thread>
#include <vector>

#include "backend.hpp"
#include "common.hpp"
#include "host_slots.hpp"

namespace mlxhip {
namespace {

constexpr size_t HUGE = size_t(2) << 20;  // a transparent huge page of the destination
// 512 KiB chunks took 1.7 times as long as 2 MiB ones (each is a transfer and
// an event of its own).
constexpr size_t CHUNK = HUGE;
constexpr size_t PAGE = 4096;
constexpr int MAX_WORKERS = 8;
constexpr size_t MIN_BYTES = size_t(128) << 10;  // below, the runtime's own staging is as fast
// Slots that a copy of several chunks needs to be ahead of the runtime's way.
constexpr int MIN_WORKERS = 4;

char* pin_slot() {
    // Not a stream operation: allowed while another thread's stream is captured.
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    const bool exchanged = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
    void* p = nullptr;
    const hipError_t e = hipHostMalloc(&p, CHUNK, hipHostMallocPortable);
    if (exchanged) (void)hipThreadExchangeStreamCaptureMode(&mode);
    if (e == hipSuccess) return static_cast<char*>(p);
    (void)hipGetLastError();
    return nullptr;
}

void unpin_slot(char* p) { (void)hipHostFree(p); }

HostSlots& slots() {
    static HostSlots* p = new HostSlots(pin_slot, unpin_slot);  // never destroyed: outlives late frees at exit
    return *p;
}

// Faults the pages of [p, p + n) in (all of them are written afterwards).
void touch(char* p, size_t n) {
    for (size_t i = 0; i < n; i += PAGE) *static_cast<volatile char*>(p + i) = 0;
}

}  // namespace

void host_copy_retain() { slots().retain(); }
void host_copy_release() { slots().release(); }

int copy_to_host(void* dst, const void* src, size_t bytes, hipStream_t s) {
    // Chunks end at 2 MiB boundaries of the destination, so that no two threads
    // fault the same huge page.
    const size_t head = bytes <= CHUNK ? bytes : CHUNK - reinterpret_cast<uintptr_t>(dst) % HUGE;
    const int chunks = 1 + (int)((bytes - head + CHUNK - 1) / CHUNK);
    char* slot[MAX_WORKERS];
    int workers = 0;
    if (bytes >= MIN_BYTES) {
        static const int cpus = (int)std::thread::hardware_concurrency();
        const int most = std::max(1, std::min({chunks, MAX_WORKERS, cpus / 2}));
        workers = slots().take(bytes, most, std::min(most, MIN_WORKERS), slot);
    }
    if (workers == 0) {
        MLXHIP_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s));
        MLXHIP_HIP(hipStreamSynchronize(s));
        return MLXHIP_OK;
    }
    char* to = static_cast<char*>(dst);
    const char* from = static_cast<const char*>(src);
    if (chunks == 1) {
        hipError_t e = hipMemcpyAsync(slot[0], from, bytes, hipMemcpyDeviceToHost, s);
        touch(to, bytes);  // while the transfer runs
        const hipError_t es = hipStreamSynchronize(s);
        if (e == hipSuccess) e = es;
        if (e == hipSuccess) std::memcpy(to, slot[0], bytes);
        slots().give(slot, 1);
        return e == hipSuccess ? MLXHIP_OK : hip_fail(e, "copy to host");
    }
    int dev = 0;
    (void)hipGetDevice(&dev);
    std::atomic<int> next{0}, error{(int)hipSuccess};
    auto work = [&](int w) noexcept {
        hipEvent_t ev = nullptr;
        hipError_t e = hipSetDevice(dev);
        if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
        while (e == hipSuccess && error.load() == (int)hipSuccess) {
            const int c = next.fetch_add(1);
            if (c >= chunks) break;
            const size_t lo = c == 0 ? 0 : head + (size_t)(c - 1) * CHUNK;
            const size_t n = std::min(bytes, head + (size_t)c * CHUNK) - lo;
            e = hipMemcpyAsync(slot[w], from + lo, n, hipMemcpyDeviceToHost, s);
            if (e == hipSuccess) e = hipEventRecord(ev, s);
            if (e == hipSuccess) touch(to + lo, n);  // while its transfer runs
            if (e == hipSuccess) e = hipEventSynchronize(ev);
            if (e == hipSuccess) std::memcpy(to + lo, slot[w], n);
        }
        if (e != hipSuccess) {
            (void)hipGetLastError();
            error.store((int)e);
        }
        if (ev) (void)hipEventDestroy(ev);
    };
    std::vector<std::thread> threads;
    try {
        threads.reserve((size_t)workers);
        for (int w = 1; w < workers; ++w) threads.emplace_back(work, w);
    } catch (const std::exception&) {
        // Fewer threads then: the chunks are handed out one by one.
    }
    work(0);
    for (std::thread& t : threads) t.join();
    const hipError_t e = (hipError_t)error.load();
    // A failed copy may leave transfers queued into the slots.
    if (e != hipSuccess) (void)hipStreamSynchronize(s);
    slots().give(slot, workers);
    return e == hipSuccess ? MLXHIP_OK : hip_fail(e, "copy to host");
}

}  // namespace mlxhip
