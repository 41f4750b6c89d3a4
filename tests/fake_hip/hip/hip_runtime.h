// The part of the HIP runtime that the readback header calls, on the host:
// several devices, streams that may never drain, pinned memory counted.
// Copies are done when they are enqueued; on a stuck stream, or to a device,
// they are only noted.  Test infrastructure.
#pragma once

#include <atomic>
#include <cstddef>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>

#define __global__
#define __device__
#define __host__
#define __launch_bounds__(...)
#define __HIP_MEMORY_SCOPE_SYSTEM 0
#define __hip_atomic_store(p, v, order, scope) __atomic_store_n(p, v, order)

struct FakeDim {
    unsigned int x = 0, y = 0, z = 0;
};
static FakeDim threadIdx;

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorInvalidHandle = 400, hipErrorNotReady = 600 };
enum hipMemcpyKind { hipMemcpyDeviceToHost = 2, hipMemcpyDefault = 4 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1, hipMemoryTypeDevice = 2, hipMemoryTypeManaged = 3 };
constexpr unsigned int hipEventDisableTiming = 2, hipHostMallocDefault = 0;

struct FakeStream {
    int device = 0;
    std::atomic<bool> stuck{false};
};
typedef FakeStream* hipStream_t;

struct FakeEvent {
    int device = 0;
    FakeStream* on = nullptr;
};
typedef FakeEvent* hipEvent_t;

struct hipPointerAttribute_t {
    hipMemoryType type = hipMemoryTypeUnregistered;
    int device = 0;
};

struct FakeRuntime {
    std::mutex m;
    std::map<char*, size_t> pinned;  // by hipHostMalloc, and what a test adds as its own
    std::map<char*, size_t> on_device;
    size_t pinned_bytes = 0;
    std::atomic<int> pins{0}, frees{0}, copies{0}, unbounded_waits{0};
    std::map<void*, size_t> copied_to;  // destinations of copies
    std::atomic<bool> no_pinning{false};
    std::atomic<int> null_stream_device{-1};  // device of the last wait on the null stream
};
inline FakeRuntime& fake() {
    static FakeRuntime r;
    return r;
}
inline thread_local int fake_device = 0;

inline bool fake_find(const std::map<char*, size_t>& in, const void* p) {
    auto it = in.upper_bound(const_cast<char*>(static_cast<const char*>(p)));
    if (it == in.begin()) return false;
    --it;
    return static_cast<const char*>(p) < it->first + it->second;
}

inline hipError_t hipGetDevice(int* d) {
    *d = fake_device;
    return hipSuccess;
}
inline hipError_t hipSetDevice(int d) {
    fake_device = d;
    return hipSuccess;
}
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t bytes, unsigned int) {
    if (fake().no_pinning) return hipErrorOutOfMemory;
    *p = std::malloc(bytes);
    std::lock_guard<std::mutex> lk(fake().m);
    fake().pinned[static_cast<char*>(*p)] = bytes;
    fake().pinned_bytes += bytes;
    fake().pins++;
    return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
    std::lock_guard<std::mutex> lk(fake().m);
    fake().pinned_bytes -= fake().pinned[static_cast<char*>(p)];
    fake().pinned.erase(static_cast<char*>(p));
    fake().frees++;
    std::free(p);
    return hipSuccess;
}
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    std::lock_guard<std::mutex> lk(fake().m);
    *a = hipPointerAttribute_t{};
    if (fake_find(fake().pinned, p)) a->type = hipMemoryTypeHost;
    else if (fake_find(fake().on_device, p)) a->type = hipMemoryTypeDevice;
    else return hipErrorInvalidValue;
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned int) {
    *e = new FakeEvent{fake_device, nullptr};
    return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
    delete e;
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    if (e->device != s->device) return hipErrorInvalidHandle;
    e->on = s;
    return hipSuccess;
}
inline hipError_t hipEventQuery(hipEvent_t e) { return e->on && e->on->stuck ? hipErrorNotReady : hipSuccess; }
inline hipError_t hipStreamQuery(hipStream_t s) { return s->stuck ? hipErrorNotReady : hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t s) {
    if (!s) {
        fake().null_stream_device = fake_device;
    } else if (s->stuck) {  // would never return
        fake().unbounded_waits++;
    }
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind, hipStream_t s) {
    fake().copies++;
    std::unique_lock<std::mutex> lk(fake().m);
    fake().copied_to[dst] = bytes;
    const bool device = fake_find(fake().on_device, dst);
    lk.unlock();
    if (!s->stuck && !device) std::memcpy(dst, src, bytes);
    return hipSuccess;
}
