// A stand-in for the HIP runtime calls of csrc/host_copy.cpp, for the CPU test
// beside it: device memory is host memory, the work of a stream is queued and
// done when something waits for it, the current device belongs to the thread,
// and calls can be made to fail.
#pragma once
#include <atomic>
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <vector>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorInvalidDevice = 101,
                  hipErrorInvalidHandle = 400 };
enum hipMemcpyKind { hipMemcpyDeviceToHost = 2 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1, hipMemoryTypeDevice = 2 };
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2;

struct hipPointerAttribute_t {
    hipMemoryType type;
    int device;
};
struct FakeCopy {
    void* dst;
    const void* src;
    size_t n;
};
struct FakeStream {
    int device = 0;
    std::mutex lock;
    std::vector<FakeCopy> queued;
    FakeStream() { queued.reserve(1024); }   // (the runtime's calls throw nothing)
};
struct FakeEvent {
    int device;
    FakeStream* on;
};
typedef FakeStream* hipStream_t;
typedef FakeEvent* hipEvent_t;
typedef int hipDevice_t;

namespace fake {
inline thread_local int current = 0;
inline std::atomic<int> events{0}, pinned{0};          // alive
inline std::atomic<int> staged{0}, plain{0};           // copies
inline std::atomic<int> event_creations_left{-1};      // then they fail (negative: never)
inline std::atomic<int> records_left{-1};
// memory that the runtime knows, with its kind
inline const char *known = nullptr, *known_end = nullptr;
inline hipMemoryType known_type = hipMemoryTypeUnregistered;
inline bool knows(const void* p)
{
    const char* c = static_cast<const char*>(p);
    return c >= known && c < known_end;
}

inline bool spent(std::atomic<int>& left) { return left >= 0 && left-- == 0; }
inline void drain(FakeStream* s)
{
    std::lock_guard<std::mutex> hold(s->lock);
    for (auto& c : s->queued) std::memcpy(c.dst, c.src, c.n);
    s->queued.clear();
}
inline size_t pending(FakeStream* s)
{
    std::lock_guard<std::mutex> hold(s->lock);
    return s->queued.size();
}
}  // namespace fake

inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int* d) { *d = fake::current; return hipSuccess; }
inline hipError_t hipSetDevice(int d) { fake::current = d; return hipSuccess; }
inline hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t* d) { *d = s->device; return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    *p = std::malloc(n);
    ++fake::pinned;
    return hipSuccess;
}
inline hipError_t hipHostFree(void* p)
{
    std::free(p);
    --fake::pinned;
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
    if (fake::spent(fake::event_creations_left)) {
        fake::event_creations_left = 0;
        return hipErrorOutOfMemory;
    }
    *e = static_cast<FakeEvent*>(std::malloc(sizeof(FakeEvent)));
    (*e)->device = fake::current;
    (*e)->on = nullptr;
    ++fake::events;
    return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e)
{
    std::free(e);
    --fake::events;
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    if (e->device != s->device) return hipErrorInvalidHandle;
    if (fake::spent(fake::records_left)) return hipErrorInvalidHandle;
    e->on = s;
    return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e)
{
    if (e->on) fake::drain(e->on);
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s)
{
    fake::drain(s);
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t s)
{
    ++fake::staged;
    std::lock_guard<std::mutex> hold(s->lock);
    s->queued.push_back(FakeCopy{dst, src, n});
    return hipSuccess;
}
inline hipError_t hipMemcpy(void* dst, const void* src, size_t n, hipMemcpyKind)
{
    ++fake::plain;   // (of the null stream: nothing of another stream is waited for)
    std::memcpy(dst, src, n);
    return hipSuccess;
}
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p)
{
    a->type = fake::knows(p) ? fake::known_type : hipMemoryTypeUnregistered;
    a->device = 0;
    return hipSuccess;
}
