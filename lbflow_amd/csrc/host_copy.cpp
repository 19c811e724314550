// host_copy.cpp -- see host_copy.h.
#include "host_copy.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

namespace lbf {

namespace {
constexpr unsigned WORKERS = 8;
constexpr size_t CHUNK = size_t(2) << 20;
// Below this the runtime's copy is as fast: starting the threads takes about
// 0.1 ms, in which it moves 1 MB, and each thread should get a few chunks.
constexpr size_t SMALL = size_t(8) << 20;
}  // namespace

class HostStage {
  public:
    explicit HostStage(int dev) : device(dev) {}
    const int device;
    std::mutex busy;   // one copy at a time uses the buffers
    char* pinned = nullptr;
    hipEvent_t done[WORKERS][2] = {};

    ~HostStage() { release(); }
    // busy held, the stage's device current
    bool ready()
    {
        if (pinned) return true;
        void* p = nullptr;
        if (hipHostMalloc(&p, WORKERS * 2 * CHUNK, hipHostMallocDefault) != hipSuccess) return false;
        pinned = static_cast<char*>(p);
        for (auto& w : done)
            for (hipEvent_t& e : w)
                if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
                    e = nullptr;
                    release();
                    return false;
                }
        return true;
    }
    char* buffer(unsigned w, int k) { return pinned + (size_t(w) * 2 + size_t(k)) * CHUNK; }

  private:
    void release()
    {
        for (auto& w : done)
            for (hipEvent_t& e : w) {
                if (e) (void)hipEventDestroy(e);
                e = nullptr;
            }
        if (pinned) (void)hipHostFree(pinned);
        pinned = nullptr;
    }
};

static std::shared_ptr<HostStage> host_stage(int dev)
{
    static std::mutex lock;
    static std::map<int, std::weak_ptr<HostStage>> stages;
    std::lock_guard<std::mutex> hold(lock);
    std::shared_ptr<HostStage> s = stages[dev].lock();
    if (!s) stages[dev] = s = std::make_shared<HostStage>(dev);
    return s;
}

namespace {
// Makes a device the calling thread's current one for a scope: events belong to
// the device that is current when they are created, and the caller's choice
// stays the caller's.
class CurrentDevice {
  public:
    explicit CurrentDevice(int dev)
    {
        if (hipGetDevice(&before) != hipSuccess) return;
        set = before == dev || hipSetDevice(dev) == hipSuccess;
        changed = set && before != dev;
    }
    ~CurrentDevice()
    {
        if (changed) (void)hipSetDevice(before);
    }
    CurrentDevice(const CurrentDevice&) = delete;
    CurrentDevice& operator=(const CurrentDevice&) = delete;
    bool set = false;

  private:
    int before = 0;
    bool changed = false;
};
}  // namespace

// The stage's device is current.
static hipError_t copy_parallel(HostStage& st, char* dst, const char* src, size_t bytes, hipStream_t s)
{
    const size_t chunks = (bytes + CHUNK - 1) / CHUNK;
    std::atomic<size_t> next{0};
    std::atomic<int> error{int(hipSuccess)};
    auto work = [&](unsigned w) {
        constexpr size_t NONE = ~size_t(0);
        size_t held[2] = {NONE, NONE};
        if (w && hipSetDevice(st.device) != hipSuccess) error = int(hipErrorInvalidDevice);   // 0: the caller's thread
        for (int cur = 0;; cur ^= 1) {
            hipError_t e = hipSuccess;
            const size_t k = error == int(hipSuccess) ? next++ : chunks;
            if (k < chunks) {
                e = hipMemcpyAsync(st.buffer(w, cur), src + k * CHUNK, std::min(CHUNK, bytes - k * CHUNK),
                                   hipMemcpyDeviceToHost, s);
                if (e == hipSuccess) e = hipEventRecord(st.done[w][cur], s);
                if (e == hipSuccess) held[cur] = k;
            }
            const int old = cur ^ 1;
            if (held[old] != NONE) {
                const size_t o = held[old] * CHUNK;
                const hipError_t f = hipEventSynchronize(st.done[w][old]);
                if (f == hipSuccess) std::memcpy(dst + o, st.buffer(w, old), std::min(CHUNK, bytes - o));
                else e = f;
                held[old] = NONE;
            }
            if (e != hipSuccess) error = int(e);
            if (held[0] == NONE && held[1] == NONE && (k >= chunks || error != int(hipSuccess))) break;
        }
    };
    const unsigned n = unsigned(std::min<size_t>({WORKERS, (chunks + 1) / 2,
                                                  std::max(1u, std::thread::hardware_concurrency())}));
    std::vector<std::thread> pool;
    pool.reserve(n);
    try {
        for (unsigned w = 1; w < n; ++w) pool.emplace_back(work, w);
    } catch (const std::exception&) {
        // no thread or no memory for one: those that did start and this one take all
        // chunks (and are joined: a std::thread that goes out of scope unjoined
        // ends the process)
    }
    work(0);
    for (std::thread& t : pool) t.join();
    // a copy whose event could not be recorded is still on its way into a buffer
    if (error != int(hipSuccess)) (void)hipStreamSynchronize(s);
    return hipError_t(error.load());
}

// Ordinary host memory is what the runtime does not know.  Into pinned memory
// its own copy is one transfer at the link's rate (57 GB/s; the threads reach
// 38 there), and device memory is not the CPU's to write.
static hipMemoryType memory_type(const void* p)
{
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type;
    (void)hipGetLastError();   // (older runtimes call unknown memory an error)
    return hipMemoryTypeUnregistered;
}

hipError_t copy_to_host(std::shared_ptr<HostStage>& stage, void* dst, const void* src, size_t bytes, hipStream_t s)
{
    hipDevice_t dev = 0;
    const hipMemoryType to = memory_type(dst);
    if (bytes >= SMALL && to == hipMemoryTypeUnregistered && hipStreamGetDevice(s, &dev) == hipSuccess) {
        try {
            const CurrentDevice current(dev);
            if (!stage) stage = host_stage(dev);
            if (current.set) {
                std::lock_guard<std::mutex> hold(stage->busy);
                if (stage->ready())
                    return copy_parallel(*stage, static_cast<char*>(dst), static_cast<const char*>(src), bytes, s);
            }
        } catch (const std::exception&) {
            // out of host memory or threads: the plain copy below
        }
    }
    if (to != hipMemoryTypeUnregistered && to != hipMemoryTypeHost) {
        // device memory: even the blocking call may return before the end
        const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
        return e != hipSuccess ? e : hipStreamSynchronize(s);
    }
    // The blocking call after the stream's work is the quickest for small results: fields of
    // 320 sites 27 us, 35 by hipMemcpyWithStream and 44 by an asynchronous copy and a wait
    // (200 steps, a report and the fields 508, 527 and 525).
    const hipError_t e = hipStreamSynchronize(s);
    return e != hipSuccess ? e : hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost);
}

}  // namespace lbf
