// Split-K partial scratch: one FP32 buffer per (device, kind), reused across calls; and the flash
// key-split scratch, one buffer per stream (StreamScratch).
// Growth rule as in the reference's src/runtime/scratch_pool.cpp:38-60 (x1.25 + 1024 elements).

#include <algorithm>
#include <cstring>
#include <map>
#include <mutex>
#include <utility>
#include <vector>

#include "device/device.hpp"
#include "runtime/internal.hpp"
#include "sca_hip.h"

namespace sca {
namespace runtime {
namespace {

struct Entry {
    void* ptr{nullptr};
    size_t elements{0};
    int device_id{0};
};

std::mutex& PoolMutex() {
    static std::mutex mu;
    return mu;
}

// Leaked on purpose: freeing device memory from a static destructor would race the HIP runtime's
// own teardown at process exit.
std::map<std::pair<int, int>, Entry>& Pool() {
    static auto* pool = new std::map<std::pair<int, int>, Entry>();
    return *pool;
}

size_t g_high_water_bytes = 0;

}  // namespace

sci::Result<float*> AcquireScratchFp32(ScratchKind kind, size_t elements, int device_id) {
    if (elements == 0) {
        return sci::MakeUnexpected<float*>(
            MakeStatus(AttnStatusCode::kWorkspaceExceeded, "scratch request with 0 elements"));
    }
    std::lock_guard<std::mutex> lock(PoolMutex());
    Entry& entry = Pool()[{device_id, static_cast<int>(kind)}];
    if (entry.ptr == nullptr || entry.elements < elements) {
        sci::Device& device = sci::GpuDevice(device_id);
        if (entry.ptr != nullptr) {
            // The previous buffer may still be read by queued kernels.
            device.synchronize();
            device.deallocate(entry.ptr);
            entry.ptr = nullptr;
            entry.elements = 0;
        }
        const size_t grown = static_cast<size_t>(static_cast<double>(elements) * 1.25) + 1024;
        entry.ptr = device.allocate(grown * sizeof(float));
        if (entry.ptr == nullptr) {
            return sci::MakeUnexpected<float*>(MakeStatus(
                AttnStatusCode::kWorkspaceExceeded,
                "scratch allocation of " + std::to_string(grown * sizeof(float)) + " B failed"));
        }
        entry.elements = grown;
        entry.device_id = device_id;
        g_high_water_bytes = std::max(g_high_water_bytes, grown * sizeof(float));
    }
    return sci::Ok(static_cast<float*>(entry.ptr));
}

namespace {

constexpr size_t kMaxStreamSlots = 4;
constexpr size_t kMaxStreamScratchBytes = size_t{64} << 20;

struct StreamSlot {
    int device_id{0};
    void* stream{nullptr};  // of the last use
    void* ptr{nullptr};
    size_t bytes{0};
    void* event{nullptr};   // recorded after the last use
    uint64_t used{0};       // order of last uses
};

std::mutex& StreamMutex() {
    static std::mutex mu;
    return mu;
}

std::vector<StreamSlot*>& StreamSlots() {  // leaked on purpose, like the scratch pool
    static auto* slots = new std::vector<StreamSlot*>();
    return *slots;
}

// Frees the buffer once its last use has completed; false when that cannot be known (it stays).
bool FreeSlotBuffer(StreamSlot* slot) {
    if (slot->ptr == nullptr) return true;
    if (slot->used != 0 && sca_hip_event_synchronize(slot->event) != 0) return false;
    sci::GpuDevice(slot->device_id).deallocate(slot->ptr);
    slot->ptr = nullptr;
    slot->bytes = 0;
    return true;
}

}  // namespace

StreamScratch::StreamScratch(size_t bytes, int device_id, void* stream) : stream_(stream) {
    if (bytes == 0 || bytes > kMaxStreamScratchBytes) return;
    int capturing = 0;
    // A graph would keep the buffer's address beyond this lease.
    if (sca_hip_stream_is_capturing(stream, &capturing) != 0 || capturing != 0) return;
    static uint64_t uses = 0;  // guarded by the mutex
    lock_ = std::unique_lock<std::mutex>(StreamMutex());
    StreamSlot* slot = nullptr;
    StreamSlot* oldest = nullptr;
    size_t on_device = 0;
    for (StreamSlot* s : StreamSlots()) {
        if (s->device_id != device_id) continue;
        ++on_device;
        if (s->stream == stream && s->used != 0) slot = s;
        if (oldest == nullptr || s->used < oldest->used) oldest = s;
    }
    if (slot == nullptr && on_device < kMaxStreamSlots) {
        slot = new StreamSlot();
        slot->device_id = device_id;
        if (sca_hip_event_create(&slot->event) != 0) {
            delete slot;
            return;
        }
        StreamSlots().push_back(slot);
    }
    if (slot == nullptr) slot = oldest;
    // Also when the handles are equal: one value can name several streams (hipStreamPerThread is a
    // stream per host thread; a handle can be reused after a destroy). On one stream the wait is free.
    if (slot->used != 0 && sca_hip_stream_wait_event(stream, slot->event) != 0) return;
    if (slot->bytes < bytes) {
        if (!FreeSlotBuffer(slot)) return;
        size_t want = size_t{1} << 20;
        while (want < bytes) want *= 2;
        slot->ptr = sci::GpuDevice(device_id).allocate(want);
        if (slot->ptr == nullptr) return;
        slot->bytes = want;
        std::lock_guard<std::mutex> pool(PoolMutex());
        g_high_water_bytes = std::max(g_high_water_bytes, want);
    }
    slot->stream = stream;
    slot->used = ++uses;
    slot_ = slot;
    ptr = slot->ptr;
}

StreamScratch::~StreamScratch() {
    if (slot_ == nullptr) return;
    StreamSlot* slot = static_cast<StreamSlot*>(slot_);
    if (sca_hip_event_record(slot->event, stream_) == 0) return;
    // The event still stands for an earlier use, which orders nothing: wait here, or give the buffer up.
    if (sca_hip_stream_synchronize(stream_) != 0) {
        slot->ptr = nullptr;
        slot->bytes = 0;
    }
}

sci::Status ReleaseScratch() {
    {
        std::lock_guard<std::mutex> streams(StreamMutex());
        for (StreamSlot* slot : StreamSlots()) (void)FreeSlotBuffer(slot);
    }
    std::lock_guard<std::mutex> lock(PoolMutex());
    for (auto& kv : Pool()) {
        if (kv.second.ptr != nullptr) {
            sci::Device& device = sci::GpuDevice(kv.second.device_id);
            device.synchronize();
            device.deallocate(kv.second.ptr);
        }
    }
    Pool().clear();
    return sci::Status::Ok();
}

size_t ScratchHighWaterMarkBytes() {
    std::lock_guard<std::mutex> lock(PoolMutex());
    return g_high_water_bytes;
}

}  // namespace runtime
}  // namespace sca

namespace sca {
namespace runtime {
namespace {

struct Staging {
    void* host{nullptr};
    size_t bytes{0};
    void* event{nullptr};  // recorded after the last copy out of `host`
};

std::mutex& StagingMutex() {
    static std::mutex mu;
    return mu;
}

std::map<int, Staging>& StagingPool() {  // leaked on purpose, like the scratch pool
    static auto* pool = new std::map<int, Staging>();
    return *pool;
}

}  // namespace

sci::Result<void*> UploadToScratch(ScratchKind kind, const void* host, size_t bytes,
                                   int device_id, void* stream) {
    sci::Result<float*> dst = AcquireScratchFp32(kind, (bytes + 3) / 4, device_id);
    if (!dst.ok()) return sci::MakeUnexpected<void*>(dst.error());
    std::lock_guard<std::mutex> lock(StagingMutex());
    Staging& st = StagingPool()[device_id];
    if (st.event != nullptr) {
        const sci::Status done =
            StatusFromHip(sca_hip_event_synchronize(st.event), "scratch staging reuse");
        if (!done.ok()) return sci::MakeUnexpected<void*>(done);
    } else {
        const sci::Status made =
            StatusFromHip(sca_hip_event_create(&st.event), "scratch staging event");
        if (!made.ok()) return sci::MakeUnexpected<void*>(made);
    }
    if (st.bytes < bytes) {
        if (st.host != nullptr) sca_hip_host_free(st.host);
        st.host = nullptr;
        st.bytes = 0;
        const size_t grown = std::max<size_t>(bytes, 4096);
        const sci::Status got =
            StatusFromHip(sca_hip_host_malloc(&st.host, grown), "scratch staging allocation");
        if (!got.ok()) return sci::MakeUnexpected<void*>(got);
        st.bytes = grown;
    }
    std::memcpy(st.host, host, bytes);
    sci::Status status = StatusFromHip(
        sca_hip_memcpy_async(*dst, st.host, bytes, SCA_COPY_H2D, stream), "scratch upload");
    if (status.ok()) {
        status = StatusFromHip(sca_hip_event_record(st.event, stream), "scratch staging event");
    }
    if (!status.ok()) return sci::MakeUnexpected<void*>(status);
    return sci::Ok(static_cast<void*>(*dst));
}

}  // namespace runtime
}  // namespace sca
