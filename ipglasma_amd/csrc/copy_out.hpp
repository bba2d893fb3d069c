// copy_out.hpp -- device-to-host copies of fields and gradients.  The including
// file brings the HIP runtime's declarations (the host test brings stand-ins).
#pragma once
#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstring>
#include <mutex>
#include <thread>

namespace {
// Device-to-host copies of fields and gradients.  A copy into pageable memory
// goes through the runtime's staging buffer on one thread, which also takes
// the page faults of a fresh destination (4 GB/s measured, 17 GB/s once the
// pages are there, against 56 GB/s into pinned memory).  Large copies go
// through kCopyThreads pinned slots instead, each with a thread and a stream:
// one slot's transfer runs beside the others' copies to the destination.  One
// set of slots per process (kCopyThreads x kCopySlot), made at the first large
// copy, used by one call at a time (another call meanwhile takes one plain
// copy on its stream) and handed back by ipg_release_cached_memory.  Only
// pageable memory goes through the slots: a pinned, device or managed
// destination takes one plain copy (the DMA writes it: T^{mu nu} at N = 256
// into pinned memory 0.10 ms, through the slots 0.19; and the slots' memcpy is
// the host's, for host memory).
constexpr int kCopyThreads = 8;
constexpr size_t kCopySlot = (size_t)2 << 20;
struct CopyPool {
    std::mutex m;
    int dev = -1;
    char* slot[kCopyThreads] = {nullptr};
    hipStream_t st[kCopyThreads] = {nullptr};
    void release() {
        for (int t = 0; t < kCopyThreads; t++) {
            if (slot[t]) (void)hipHostFree(slot[t]);
            if (st[t]) (void)hipStreamDestroy(st[t]);
            slot[t] = nullptr;
            st[t] = nullptr;
        }
        dev = -1;
    }
    bool ready(int d) {
        if (dev == d) return true;
        release();
        for (int t = 0; t < kCopyThreads; t++)
            if (hipHostMalloc((void**)&slot[t], kCopySlot, hipHostMallocDefault) != hipSuccess ||
                hipStreamCreateWithFlags(&st[t], hipStreamNonBlocking) != hipSuccess) {
                (void)hipGetLastError();
                release();
                return false;
            }
        dev = d;
        return true;
    }
};
// never destroyed, as the block cache
CopyPool& copy_pool() {
    static CopyPool* p = new CopyPool;
    return *p;
}
// One copy on the caller's stream: hipMemcpy goes to the null stream, which
// waits for every other context's stream and holds up their next work.
hipError_t copy_plain(void* dst, const void* src, size_t n, hipStream_t st) {
    return hipMemcpyWithStream(dst, src, n, hipMemcpyDefault, st);
}
bool pageable(const void* p) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
    (void)hipGetLastError();  // runtimes that know nothing of pageable memory
    return true;
}
// n bytes from device memory, after the work queued on `after`
hipError_t copy_out(void* dst, const void* src, size_t n, hipStream_t after) {
    if (n < 2 * kCopySlot || !pageable(dst)) return copy_plain(dst, src, n, after);
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    // the slots' streams do not wait for the others by themselves
    if (e == hipSuccess) e = hipStreamSynchronize(after);
    if (e != hipSuccess) return e;
    CopyPool& p = copy_pool();
    std::unique_lock<std::mutex> lk(p.m, std::try_to_lock);
    if (!lk.owns_lock() || !p.ready(dev)) return copy_plain(dst, src, n, after);
    const size_t chunks = (n + kCopySlot - 1) / kCopySlot;
    const int nt = (int)std::min<size_t>(kCopyThreads, chunks);
    std::atomic<size_t> next{0};
    std::atomic<int> err{(int)hipSuccess};
    auto work = [&](int t) {
        if (hipSetDevice(dev) != hipSuccess) {
            err = (int)hipErrorInvalidDevice;
            return;
        }
        for (size_t c = next++; c < chunks && err == (int)hipSuccess; c = next++) {
            const size_t o = c * kCopySlot, len = std::min(kCopySlot, n - o);
            hipError_t r = hipMemcpyAsync(p.slot[t], (const char*)src + o, len, hipMemcpyDeviceToHost, p.st[t]);
            if (r == hipSuccess) r = hipStreamSynchronize(p.st[t]);
            if (r != hipSuccess) {
                err = (int)r;
                return;
            }
            std::memcpy((char*)dst + o, p.slot[t], len);
        }
    };
    std::thread th[kCopyThreads];
    try {
        for (int t = 1; t < nt; t++) th[t] = std::thread(work, t);
    } catch (...) {
        // fewer threads: the others take the chunks
    }
    work(0);
    for (std::thread& x : th)
        if (x.joinable()) x.join();
    return (hipError_t)err.load();
}
// hands the slots back; waits for a copy that is using them
void copy_out_release() {
    CopyPool& p = copy_pool();
    std::lock_guard<std::mutex> lk(p.m);
    p.release();
}
}  // namespace
