// copy_out of ipglasma_amd/csrc/copy_out.hpp on a stand-in for the HIP runtime:
// "device" memory is host memory, a copy queued on a stream runs when that
// stream is synchronised, and a copy on the null stream first drains every
// blocking stream, as the runtime's does.
#include <algorithm>
#include <cstdlib>
#include <functional>
#include <map>
#include <mutex>
#include <vector>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorInvalidDevice = 101 };
enum hipMemcpyKind { hipMemcpyDeviceToHost = 2, hipMemcpyDefault = 4 };
enum hipMemoryType {
    hipMemoryTypeUnregistered = 0,
    hipMemoryTypeHost = 1,
    hipMemoryTypeDevice = 2,
    hipMemoryTypeManaged = 3
};
struct hipPointerAttribute_t {
    hipMemoryType type;
};
constexpr unsigned hipHostMallocDefault = 0, hipStreamNonBlocking = 1;
struct Stream {
    bool blocking;
    std::vector<std::function<void()>> q;
};
typedef Stream* hipStream_t;

namespace {
std::recursive_mutex rt;  // one runtime lock
hipError_t last = hipSuccess;
std::vector<Stream*> blocking;
const char* dst_lo = nullptr;
size_t dst_n = 0;
long long null_copies, direct_bytes, slot_bytes, slot_copies, live_slots, live_streams;
int dst_kind, fail_mode;

hipError_t err(hipError_t e) {
    if (e != hipSuccess) last = e;
    return e;
}
void drain(Stream* s) {
    for (auto& f : s->q) f();
    s->q.clear();
}
}  // namespace

hipError_t hipGetLastError() {
    std::lock_guard<std::recursive_mutex> lk(rt);
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    std::lock_guard<std::recursive_mutex> lk(rt);
    if (fail_mode == 1 && live_slots == 3) return err(hipErrorOutOfMemory);
    live_slots++;
    *p = std::malloc(n);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    std::lock_guard<std::recursive_mutex> lk(rt);
    live_slots--;
    std::free(p);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    std::lock_guard<std::recursive_mutex> lk(rt);
    live_streams++;
    *s = new Stream{false, {}};
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    std::lock_guard<std::recursive_mutex> lk(rt);
    live_streams--;
    delete s;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    std::lock_guard<std::recursive_mutex> lk(rt);
    drain(s);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    std::lock_guard<std::recursive_mutex> lk(rt);
    const bool known = (const char*)p >= dst_lo && (const char*)p < dst_lo + dst_n && dst_kind != 0;
    if (!known && fail_mode == 3) return err(hipErrorInvalidValue);  // runtimes that know no pageable pointer
    a->type = known ? (hipMemoryType)dst_kind : hipMemoryTypeUnregistered;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
    std::lock_guard<std::recursive_mutex> lk(rt);
    const bool direct = (char*)d >= dst_lo && (char*)d < dst_lo + dst_n;
    (direct ? direct_bytes : slot_bytes) += (long long)n;
    if (!direct && fail_mode == 2 && ++slot_copies == 4) return err(hipErrorInvalidValue);
    st->q.push_back([=] { __builtin_memcpy(d, s, n); });
    return hipSuccess;
}
hipError_t hipMemcpyWithStream(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t st) {
    std::lock_guard<std::recursive_mutex> lk(rt);
    const hipError_t e = hipMemcpyAsync(d, s, n, k, st);
    return e == hipSuccess ? hipStreamSynchronize(st) : e;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    std::lock_guard<std::recursive_mutex> lk(rt);
    null_copies++;
    for (Stream* b : blocking) drain(b);
    __builtin_memcpy(d, s, n);
    return hipSuccess;
}

#include "../../ipglasma_amd/csrc/copy_out.hpp"

// One copy of n bytes whose source is written by work queued on the context's
// stream, while another context's stream has work queued.  kind: of the
// destination (hipMemoryType); busy: another caller holds the slots; fail: 1
// no pinned memory, 2 a slot's copy fails, 3 the runtime knows no pageable
// pointer.  out: status, destination right, another stream drained, null
// stream copies, bytes copied straight to the destination, bytes through
// slots, the error left behind, slots and streams alive after the release.
extern "C" void copy_out_case(long long n, int kind, int busy, int fail, long long* out) {
    null_copies = direct_bytes = slot_bytes = slot_copies = 0;
    last = hipSuccess;
    dst_kind = kind;
    fail_mode = fail;
    std::vector<unsigned char> src(n, 0), dst(n, 0xEE);
    dst_lo = (const char*)dst.data();
    dst_n = (size_t)n;
    Stream mine{true, {}}, other{true, {}};
    blocking = {&mine, &other};
    auto byte = [](long long i) { return (unsigned char)((i * 2654435761u) >> 13); };
    mine.q.push_back([&] {
        for (long long i = 0; i < n; i++) src[i] = byte(i);
    });
    bool drained = false;
    other.q.push_back([&] { drained = true; });
    if (busy) copy_pool().m.lock();
    hipError_t e = hipSuccess;
    std::thread t([&] { e = copy_out(dst.data(), src.data(), (size_t)n, &mine); });
    t.join();
    if (busy) copy_pool().m.unlock();
    bool ok = true;
    for (long long i = 0; i < n && ok; i++) ok = dst[i] == byte(i);
    out[0] = e;
    out[1] = ok;
    out[2] = drained;
    out[3] = null_copies;
    out[4] = direct_bytes;
    out[5] = slot_bytes;
    out[6] = hipGetLastError();
    copy_out_release();
    out[7] = live_slots + live_streams;
    blocking.clear();
}
extern "C" long long copy_out_slot() { return (long long)kCopySlot; }
