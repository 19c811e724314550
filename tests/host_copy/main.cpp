// One scenario of csrc/host_copy.cpp on the stand-in runtime of hip/hip_runtime.h;
// exit status 0 if it holds.  Every wrong result prints a line.
#include "host_copy.h"

#include <cstdio>
#include <cstdint>
#include <new>
#include <vector>
#include <string>

// The allocation that fails: the n-th of the main thread from now on (negative: none).
static thread_local int news_left = -1;
void* operator new(size_t n)
{
    if (news_left >= 0 && news_left-- == 0) throw std::bad_alloc();
    if (void* p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

static int wrong = 0;
static void check(bool ok, const char* what)
{
    if (ok) return;
    std::printf("wrong: %s\n", what);
    ++wrong;
}

struct Data {
    std::vector<char> src, dst;
    explicit Data(size_t n) : src(n), dst(n, 0)
    {
        for (size_t i = 0; i < n; ++i) src[i] = char(i * 2654435761u >> 13);
    }
    bool arrived() const { return src == dst; }
};

static hipError_t copy(std::shared_ptr<lbf::HostStage>& stage, Data& d, hipStream_t s)
{
    return lbf::copy_to_host(stage, d.dst.data(), d.src.data(), d.src.size(), s);
}

// A copy on a stream of another device than the caller's current one, as the first copy on
// that device and as a later one.
static void other_device()
{
    FakeStream s;
    s.device = 1;
    std::shared_ptr<lbf::HostStage> first, later;
    for (int current : {0, 1, 0}) {
        for (auto* stage : {&first, &later}) {
            Data d((size_t(20) << 20) + 12345);
            fake::current = current;
            check(copy(*stage, d, &s) == hipSuccess, "the copy succeeds");
            check(d.arrived(), "the data arrive");
            check(fake::current == current, "the caller's device is still current");
        }
    }
    check(first == later && first, "one stage serves the device");
}

// An allocation of the calling thread fails, each one of the copy's in turn: while the
// handle is taken, between the threads that start, after them.
static void no_memory()
{
    FakeStream s;
    for (int n = 0; n < 16; ++n) {
        std::shared_ptr<lbf::HostStage> stage;
        Data d((size_t(40) << 20) + 1);
        news_left = n;
        const hipError_t e = copy(stage, d, &s);
        news_left = -1;
        check(e == hipSuccess && d.arrived(), "the data arrive");
    }
}

// The creation of an event fails: the plain copy serves, nothing made on the way stays
// behind, and a later copy finds the stage whole.
static void no_event()
{
    FakeStream s;
    for (int n : {0, 1, 7, 15}) {
        std::shared_ptr<lbf::HostStage> stage;
        fake::event_creations_left = n;
        Data d(size_t(9) << 20);
        check(copy(stage, d, &s) == hipSuccess && d.arrived(), "the plain copy serves");
        check(fake::events == 0 && fake::pinned == 0, "what was made is given back");
        fake::event_creations_left = -1;
        Data e(size_t(9) << 20);
        check(copy(stage, e, &s) == hipSuccess && e.arrived(), "a later copy serves");
        check(fake::events == 16 && fake::pinned == 1, "one set of events and buffers");
        stage.reset();
        check(fake::events == 0 && fake::pinned == 0, "released with the last handle");
    }
}

// An event cannot be recorded behind a copy that is already queued: the call reports it
// after that copy is done, since the next call fills the same buffers.
static void no_record()
{
    FakeStream s;
    for (int n : {0, 3, 9}) {
        std::shared_ptr<lbf::HostStage> stage;
        fake::records_left = n;
        Data d((size_t(40) << 20) + 77);
        check(copy(stage, d, &s) != hipSuccess, "the failure is reported");
        check(fake::pending(&s) == 0, "no copy into the buffers is left in flight");
        fake::records_left = -1;
        Data e((size_t(40) << 20) + 77);
        check(copy(stage, e, &s) == hipSuccess && e.arrived(), "a later copy serves");
    }
}

// Below the size from which threads help: one blocking call of the runtime.
static void small()
{
    FakeStream s;
    for (size_t n : {size_t(1), size_t(4096), (size_t(8) << 20) - 1}) {
        std::shared_ptr<lbf::HostStage> stage;
        fake::plain = fake::staged = 0;
        Data d(n), newer(n);
        newer.src[0] = char(~newer.src[0]);
        s.queued.push_back(FakeCopy{d.src.data(), newer.src.data(), n});   // work of the stream that writes the source
        check(copy(stage, d, &s) == hipSuccess && d.arrived() && d.dst[0] == newer.src[0], "the stream's results arrive");
        check(fake::plain == 1 && fake::staged == 0, "by one blocking call");
        check(!stage && fake::pinned == 0, "without a stage");
    }
}

// A destination that the runtime knows: pinned memory, which the device writes by itself,
// and device memory, which the CPU must not write.
static void known_memory()
{
    FakeStream s;
    for (hipMemoryType type : {hipMemoryTypeHost, hipMemoryTypeDevice}) {
        std::shared_ptr<lbf::HostStage> stage;
        fake::plain = fake::staged = 0;
        Data d((size_t(20) << 20) + 5);
        fake::known_type = type;
        fake::known = d.dst.data();
        fake::known_end = fake::known + d.dst.size();
        check(copy(stage, d, &s) == hipSuccess && d.arrived(), "the data have arrived");
        check(fake::plain + fake::staged == 1, "by the runtime's own copy, in one piece");
        fake::staged = 0;
        fake::known = fake::known_end = nullptr;
        Data e((size_t(20) << 20) + 5);
        check(copy(stage, e, &s) == hipSuccess && e.arrived() && fake::staged > 1, "ordinary memory through the threads");
    }
}

int main(int argc, char** argv)
{
    const std::string name = argc > 1 ? argv[1] : "";
    if (name == "other_device") other_device();
    else if (name == "no_memory") no_memory();
    else if (name == "no_event") no_event();
    else if (name == "no_record") no_record();
    else if (name == "small") small();
    else if (name == "known_memory") known_memory();
    else check(false, "unknown scenario");
    return wrong != 0;
}
