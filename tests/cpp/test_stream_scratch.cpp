// Ordering of the flash key-split scratch (runtime::StreamScratch) without a GPU: the HIP calls that
// scratch_pool.cpp makes are replaced by a log, and the checks read who waits for what. Compiled with
// src/runtime/scratch_pool.cpp and src/api/status.cpp by tests/test_stream_scratch.py.

#include <cstdio>
#include <cstdlib>
#include <string>
#include <thread>
#include <vector>

#include "device/device.hpp"
#include "runtime/internal.hpp"

namespace {
std::vector<std::string> calls;  // one entry per call, in order
bool capturing = false, record_fails = false, sync_fails = false, alloc_fails = false;
int events = 0, live = 0;

std::string Id(const void* p) { return std::to_string(reinterpret_cast<uintptr_t>(p)); }
void* Handle(uintptr_t v) { return reinterpret_cast<void*>(v); }

class FakeGpu final : public sci::Device {
public:
    sci::DeviceType type() const override { return sci::DeviceType::kGPU; }
    std::string name() const override { return "fake"; }
    void* allocate(size_t bytes) override {
        if (alloc_fails) return nullptr;
        ++live;
        return std::malloc(bytes);
    }
    void deallocate(void* ptr) override {
        calls.push_back("free " + Id(ptr));
        --live;
        std::free(ptr);
    }
    void copy_to_device(void*, const void*, size_t) override {}
    void copy_to_host(void*, const void*, size_t) override {}
    void copy_within(void*, const void*, size_t) override {}
    void memset(void*, int, size_t) override {}
    void synchronize() override {}
    void copy_async(void*, const void*, size_t, sci::Stream&) override {}
};
}  // namespace

namespace sci {
Device& GpuDevice(int) {
    static FakeGpu gpu;
    return gpu;
}
}  // namespace sci

extern "C" {
const char* sca_hip_last_error_string(void) { return "fake"; }
int sca_hip_stream_is_capturing(void*, int* out) {
    *out = capturing ? 1 : 0;
    return 0;
}
int sca_hip_stream_wait_event(void* stream, void* event) {
    calls.push_back("wait " + Id(stream) + " for " + Id(event));
    return 0;
}
int sca_hip_stream_synchronize(void* stream) {
    calls.push_back("sync " + Id(stream));
    return sync_fails ? 1 : 0;
}
int sca_hip_event_create(void** event) {
    *event = Handle(1000 + ++events);
    return 0;
}
int sca_hip_event_record(void* event, void* stream) {
    calls.push_back("record " + Id(event) + " on " + Id(stream));
    return record_fails ? 1 : 0;
}
int sca_hip_event_synchronize(void* event) {
    calls.push_back("event sync " + Id(event));
    return 0;
}
int sca_hip_host_malloc(void**, size_t) { return 1; }
int sca_hip_host_free(void*) { return 0; }
int sca_hip_memcpy_async(void*, const void*, size_t, int, void*) { return 1; }
}

namespace {
int failures = 0;
void Check(bool ok, const char* what) {
    std::printf("%s %s\n", ok ? "ok  " : "FAIL", what);
    if (!ok) ++failures;
}
bool Saw(const std::string& entry) {
    for (const std::string& c : calls) {
        if (c == entry) return true;
    }
    return false;
}
// One lease; returns its buffer and leaves the calls it made while taking it in `calls`.
void* Lease(size_t bytes, uintptr_t stream) {
    calls.clear();
    const sca::runtime::StreamScratch s(bytes, 0, Handle(stream));
    return s.ptr;
}
}  // namespace

int main() {
    constexpr size_t kMiB = size_t{1} << 20;

    // 1. One handle value, two threads: 2 is hipStreamPerThread, a different stream in each.
    void *a = nullptr, *b = nullptr;
    std::thread([&] { a = Lease(kMiB, 2); }).join();
    Check(a != nullptr && Saw("record 1001 on 2"), "a lease records its event");
    std::thread([&] { b = Lease(kMiB, 2); }).join();
    Check(b != a || Saw("wait 2 for 1001"),
          "the next lease of the same buffer waits for the event, also under an equal handle");

    // 2. Other streams get buffers of their own, at most four; the fifth waits for the oldest.
    std::vector<void*> got{b};
    for (uintptr_t s : {10, 11, 12}) got.push_back(Lease(kMiB, s));
    for (size_t i = 0; i < got.size(); ++i) {
        for (size_t j = 0; j < i; ++j) Check(got[i] != got[j], "streams do not share while there are four");
    }
    void* fifth = Lease(kMiB, 13);
    Check(fifth == b && Saw("wait 13 for 1001"), "a fifth stream waits for the oldest buffer");

    // 3. A buffer grows only after its last use has completed.
    void* grown = Lease(3 * kMiB, 13);
    Check(grown != nullptr && Saw("event sync 1001") && Saw("free " + Id(fifth)),
          "growth waits before it frees");

    // 4. No scratch: above the bound, while capturing, when the allocation fails.
    Check(Lease(65 * kMiB, 10) == nullptr, "none above 64 MiB");
    capturing = true;
    Check(Lease(kMiB, 10) == nullptr, "none for a capturing stream");
    capturing = false;
    alloc_fails = true;
    Check(Lease(8 * kMiB, 10) == nullptr, "none when the allocation fails");
    alloc_fails = false;
    Check(Lease(kMiB, 10) != nullptr, "and again afterwards");

    // 5. An event that was not recorded orders nothing: the lease ends synchronised, and a buffer
    //    whose work may still run is never handed out or freed again.
    record_fails = true;
    void* c = Lease(kMiB, 11);
    Check(c == got[2] && Saw("sync 11"), "a failed record synchronises the stream");
    sync_fails = true;
    void* lost = Lease(kMiB, 11);
    record_fails = sync_fails = false;
    void* fresh = Lease(kMiB, 11);
    Check(lost == c && fresh != nullptr && fresh != lost && !Saw("free " + Id(lost)),
          "a buffer that could not be ordered is given up");

    // 6. Released: every buffer but the one given up.
    (void)sca::runtime::ReleaseScratch();
    Check(live == 1, "release frees the buffers");
    Check(Lease(kMiB, 12) != nullptr, "a lease after the release");
    std::printf("%d failure(s)\n", failures);
    return failures == 0 ? 0 : 1;
}
