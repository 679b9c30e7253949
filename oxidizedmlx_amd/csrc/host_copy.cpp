// host_copy.cpp — copies of large results into the caller's pageable memory
// (Stream::get_buffer, crates/mlx-core/src/backend.rs:162-164, and the
// decoder's logits).
//
// hipMemcpy into pageable memory goes through the runtime's staging with one
// thread, which also takes the page faults of a fresh destination: 17 GB/s on
// memory that is already mapped, about 10 GB/s on new memory, where the link
// carries 55 GB/s into pinned memory. Here several threads each move chunks
// through a pinned slot of their own, so one chunk's copy by the CPU (and its
// page faults) runs beside the others' transfers. Into a new numpy array:
// 64 MiB 6.3 -> 1.9 ms, 16 MiB 0.94 -> 0.60 ms, 4 MiB 246 -> 205 us, 1 MiB
// 430 -> 77 us (one thread).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

#include "backend.hpp"
#include "common.hpp"

namespace mlxhip {
namespace {

constexpr size_t HUGE = size_t(2) << 20;  // a transparent huge page of the destination
// 512 KiB chunks took 1.7 times as long as 2 MiB ones (each is a transfer and
// an event of its own).
constexpr size_t CHUNK = HUGE;
constexpr size_t PAGE = 4096;
constexpr int MAX_WORKERS = 8;
constexpr size_t STAGE_BYTES = CHUNK * MAX_WORKERS;
constexpr size_t MIN_BYTES = size_t(128) << 10;  // below, the runtime's own staging is as fast

// Pinned stages kept for the next copy while any Stream or decoder lives (at
// most MAX_KEPT; concurrent copies beyond that allocate and free their own).
constexpr size_t MAX_KEPT = 2;
std::mutex g_mu;
std::vector<char*> g_kept;
int g_owners = 0;

char* take_stage() {
    {
        std::lock_guard<std::mutex> g(g_mu);
        if (!g_kept.empty()) {
            char* p = g_kept.back();
            g_kept.pop_back();
            return p;
        }
    }
    void* p = nullptr;
    if (hipHostMalloc(&p, STAGE_BYTES, hipHostMallocPortable) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    return static_cast<char*>(p);
}

void give_stage(char* p) {
    {
        std::lock_guard<std::mutex> g(g_mu);
        if (g_owners > 0 && g_kept.size() < MAX_KEPT) {
            g_kept.push_back(p);
            return;
        }
    }
    (void)hipHostFree(p);
}

}  // namespace

void host_copy_retain() {
    std::lock_guard<std::mutex> g(g_mu);
    ++g_owners;
}

void host_copy_release() {
    std::vector<char*> drop;
    {
        std::lock_guard<std::mutex> g(g_mu);
        if (--g_owners == 0) drop.swap(g_kept);
    }
    for (char* p : drop) (void)hipHostFree(p);
}

int copy_to_host(void* dst, const void* src, size_t bytes, hipStream_t s) {
    char* stage = bytes >= MIN_BYTES ? take_stage() : nullptr;
    if (!stage) {
        MLXHIP_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s));
        MLXHIP_HIP(hipStreamSynchronize(s));
        return MLXHIP_OK;
    }
    int dev = 0;
    (void)hipGetDevice(&dev);
    char* to = static_cast<char*>(dst);
    const char* from = static_cast<const char*>(src);
    // Chunks end at 2 MiB boundaries of the destination, so that no two threads
    // fault the same huge page.
    const size_t head = bytes <= CHUNK ? bytes : CHUNK - reinterpret_cast<uintptr_t>(dst) % HUGE;
    const int chunks = 1 + (int)((bytes - head + CHUNK - 1) / CHUNK);
    std::atomic<int> next{0}, error{(int)hipSuccess};
    auto work = [&](int w) noexcept {
        hipEvent_t ev = nullptr;
        hipError_t e = hipSetDevice(dev);
        if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
        char* slot = stage + (size_t)w * CHUNK;
        while (e == hipSuccess && error.load() == (int)hipSuccess) {
            const int c = next.fetch_add(1);
            if (c >= chunks) break;
            const size_t lo = c == 0 ? 0 : head + (size_t)(c - 1) * CHUNK;
            const size_t n = std::min(bytes, head + (size_t)c * CHUNK) - lo;
            e = hipMemcpyAsync(slot, from + lo, n, hipMemcpyDeviceToHost, s);
            if (e == hipSuccess) e = hipEventRecord(ev, s);
            // Fault the chunk's pages in while its transfer runs (all of it is
            // written below).
            if (e == hipSuccess)
                for (size_t i = 0; i < n; i += PAGE) *static_cast<volatile char*>(to + lo + i) = 0;
            if (e == hipSuccess) e = hipEventSynchronize(ev);
            if (e == hipSuccess) std::memcpy(to + lo, slot, n);
        }
        if (e != hipSuccess) {
            (void)hipGetLastError();
            error.store((int)e);
        }
        if (ev) (void)hipEventDestroy(ev);
    };
    const int cpus = (int)std::thread::hardware_concurrency();
    const int workers = std::max(1, std::min({chunks, MAX_WORKERS, cpus / 2}));
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
    // A failed copy may leave transfers queued into the stage.
    if (e != hipSuccess) (void)hipStreamSynchronize(s);
    give_stage(stage);
    return e == hipSuccess ? MLXHIP_OK : hip_fail(e, "copy to host");
}

}  // namespace mlxhip
