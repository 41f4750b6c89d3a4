// msim_read.hpp — device-to-host readback through a handle's own pinned
// buffers, and the bounded wait the entry points share.
//
// A copy into the caller's (pageable) memory goes through the runtime's
// staging buffer, copied out by one thread which also takes
// the page faults of a fresh array: 64 MB of entities took 6.1 ms, 10 GB/s,
// where the link moves 56 GB/s.  Here several threads each bring pieces into
// pinned slots of their own and copy them out, so link, copies and page faults
// overlap.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <thread>
#include <vector>

namespace msim {

// A handle's mailbox in pinned host memory: the device-side fault word under
// the number of the report that sent it.  A report is the last work of its
// stream so far and its store a release at system scope, so whoever reads its
// number sees what all earlier work wrote.  (Copying the word back instead is
// a transfer of its own, and asking the runtime whether the stream is done
// makes it send the GPU a marker first; 10k agents, one sync after a move
// dispatch: 36 us by a blocking copy, 27 by a report and asking, 17 by a
// report alone.)
struct Mailbox {
    unsigned long long word;  // report << 32 | fault bits
};

static __global__ __launch_bounds__(64) void k_report(const unsigned int* __restrict__ faults, Mailbox* box,
                                                      unsigned int report) {
    if (threadIdx.x == 0) {
        __hip_atomic_store(&box->word, static_cast<unsigned long long>(report) << 32 | *faults, __ATOMIC_RELEASE,
                           __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// Spins for the report, at most 200 us; false: not there yet, or never (the
// caller then waits on the stream, which also tells of errors).
inline bool await_report(const Mailbox* box, unsigned int report) {
    const auto t0 = std::chrono::steady_clock::now();
    for (uint32_t k = 1;; k++) {
        if (static_cast<unsigned int>(__atomic_load_n(&box->word, __ATOMIC_ACQUIRE) >> 32) == report) return true;
        if (k % 16u == 0u && std::chrono::steady_clock::now() - t0 > std::chrono::microseconds(200)) return false;
    }
}

// One array to read: bytes from device memory src to host memory dst.
struct ReadPart {
    void* dst;
    const void* src;
    size_t bytes;
};

// Polls `busy` (hipErrorNotReady while there is work left) until it ends or
// watchdog_ms passed (hipErrorNotReady).  Short waits spin: a sleep of 20 us
// takes about 70.
template <class Busy>
hipError_t bounded_wait(uint32_t watchdog_ms, Busy&& busy) {
    const auto t0 = std::chrono::steady_clock::now();
    for (;;) {
        const hipError_t e = busy();
        if (e != hipErrorNotReady) {
            return e;
        }
        const auto us =
            std::chrono::duration_cast<std::chrono::microseconds>(std::chrono::steady_clock::now() - t0).count();
        if (us > static_cast<long long>(watchdog_ms) * 1000) {
            return e;
        }
        if (us > 200) {
            std::this_thread::sleep_for(std::chrono::microseconds(us < 10000 ? 20 : (us < 200000 ? 50 : 500)));
        }
    }
}

// Makes a device the calling thread's current one, for as long as it lives.
// Events, pinned memory and the null stream belong to the device that is
// current, which need not be the handle's.
class DeviceScope {
public:
    explicit DeviceScope(int device) {
        if (hipGetDevice(&before_) != hipSuccess) before_ = device;
        if (before_ != device) (void)hipSetDevice(device);
        device_ = device;
    }
    ~DeviceScope() {
        if (before_ != device_) (void)hipSetDevice(before_);
    }
    DeviceScope(const DeviceScope&) = delete;
    DeviceScope& operator=(const DeviceScope&) = delete;

private:
    int before_ = 0, device_ = 0;
};

class ReadBack {
public:
    // The handle's device and stream.
    void on(int device, hipStream_t stream) {
        device_ = device;
        stream_ = stream;
    }

    // 64 MB of entities, two slots a thread, ms: slots of 0.5 MB 3.2 (every
    // transfer has a fixed cost), 1 MB 2.3, 2 MB 1.9, 4 MB 2.0; 4 threads 1.97,
    // 6 1.91, 8 1.94.
    static constexpr size_t kSlot = size_t{2} << 20;

    // Pinned memory that kernels may write `bytes` of results to directly
    // (null past one slot): no transfer follows the kernel.
    void* small(size_t bytes) {
        const DeviceScope scope(device_);
        if (bytes > kSlot || !idle() || !reserve(1)) return nullptr;
        writing_ = true;
        return slots_;
    }
    static constexpr uint32_t kThreads = 6;

    ReadBack() = default;
    ReadBack(const ReadBack&) = delete;
    ReadBack& operator=(const ReadBack&) = delete;
    ~ReadBack() {
        for (hipEvent_t e : events_) {
            (void)hipEventDestroy(e);
        }
        if (slots_) (void)hipHostFree(slots_);
    }

    // Reads the parts in stream order.  ready() waits for the stream (and
    // whatever else must hold before the caller's memory is written) and
    // returns 0, or a code that is passed on.  Otherwise returns 0, or -1 with
    // *err set (hipErrorNotReady: the watchdog expired).  After a failure the
    // slots are left alone until the stream has drained (idle).
    template <class Ready>
    int read(const std::vector<ReadPart>& parts, uint32_t watchdog_ms, hipError_t* err, Ready&& ready) {
        const DeviceScope scope(device_);
        size_t total = 0;
        for (const ReadPart& p : parts) total += p.bytes;
        std::vector<ReadPart> known, rest;
        for (const ReadPart& p : parts) (by_runtime(p, total) ? known : rest).push_back(p);
        int rc = rest.empty() && !known.empty() ? ready() : read_parts(rest, watchdog_ms, err, ready);
        if (rc == 0 && !known.empty()) rc = read_known(known, watchdog_ms, err);
        if (rc == 0) {
            writing_ = false;
        } else if (rc == -1 && *err != hipErrorNotReady) {
            (void)bounded_wait(watchdog_ms, [&] { return hipStreamQuery(stream_); });
        }
        return rc;
    }

private:
    // Where the runtime copies by itself: device memory (of any size), and
    // memory that the caller has pinned when the results do not fit one slot:
    // 64 MB of entities at 54 GB/s, 37 through the slots; 640 KB take 43 us
    // against 39.
    bool by_runtime(const ReadPart& p, size_t total) const {
        if (!p.bytes) return false;
        const hipMemoryType first = memory_type(p.dst);
        if (first == hipMemoryTypeUnregistered) return false;
        return first == memory_type(static_cast<const char*>(p.dst) + p.bytes - 1) &&
               (first == hipMemoryTypeDevice || total > kSlot);
    }

    static hipMemoryType memory_type(const void* p) {
        hipPointerAttribute_t a{};
        if (hipPointerGetAttributes(&a, p) != hipSuccess) {
            (void)hipGetLastError();
            return hipMemoryTypeUnregistered;
        }
        return a.type;
    }

    int read_known(const std::vector<ReadPart>& parts, uint32_t watchdog_ms, hipError_t* err) {
        writing_ = true;  // src may lie in a slot
        for (const ReadPart& p : parts) {
            *err = hipMemcpyAsync(p.dst, p.src, p.bytes, hipMemcpyDefault, stream_);
            if (*err != hipSuccess) return -1;
        }
        *err = bounded_wait(watchdog_ms, [&] { return hipStreamQuery(stream_); });
        return *err == hipSuccess ? 0 : -1;
    }

    template <class Ready>
    int read_parts(const std::vector<ReadPart>& parts, uint32_t watchdog_ms, hipError_t* err, Ready&& ready) {
        size_t total = 0;
        bool there = !parts.empty();
        for (const ReadPart& p : parts) {
            total += (p.bytes + 255) / 256 * 256;
            there = there && slots_ && p.src >= slots_ && p.src < slots_ + kSlot;
        }
        *err = hipSuccess;
        if (there) {  // written to small() by a kernel
            const int rc = ready();
            for (const ReadPart& p : parts) {
                if (!rc) std::memcpy(p.dst, p.src, p.bytes);
            }
            return rc;
        }
        if (total <= kSlot) {  // everything through one slot, one wait
            if (!idle() || !reserve(1)) return direct(parts, err, ready);
            writing_ = true;
            size_t at = 0;
            for (const ReadPart& p : parts) {
                if (!p.bytes) continue;
                *err = hipMemcpyAsync(slots_ + at, p.src, p.bytes, hipMemcpyDeviceToHost, stream_);
                if (*err != hipSuccess) return -1;
                at += (p.bytes + 255) / 256 * 256;
            }
            const int rc = ready();
            if (rc) return rc;
            at = 0;
            for (const ReadPart& p : parts) {
                if (!p.bytes) continue;
                std::memcpy(p.dst, slots_ + at, p.bytes);
                at += (p.bytes + 255) / 256 * 256;
            }
            return 0;
        }
        // one thread per slot's worth, two slots each
        const uint32_t n = static_cast<uint32_t>(std::min<size_t>(kThreads, std::max<size_t>(1, total / kSlot)));
        if (!idle() || !reserve(2 * n)) return direct(parts, err, ready);
        const int rc = ready();
        if (rc) return rc;
        writing_ = true;
        std::vector<Piece> pieces;
        for (const ReadPart& p : parts) {
            for (size_t o = 0; o < p.bytes; o += kSlot) {
                pieces.push_back({static_cast<char*>(p.dst) + o, static_cast<const char*>(p.src) + o,
                                  std::min(kSlot, p.bytes - o)});
            }
        }
        std::atomic<size_t> next{0};
        std::atomic<int> fault{static_cast<int>(hipSuccess)};
        auto work = [&](uint32_t t) {
            if (t) (void)hipSetDevice(device_);  // a new thread starts on device 0
            Piece held[2] = {};
            int in = 0;
            for (;;) {
                const size_t k = next.fetch_add(1);
                Piece& mine = held[in];
                mine = Piece{};
                hipError_t e = hipSuccess;
                if (k < pieces.size() && fault.load() == hipSuccess) {
                    mine = pieces[k];
                    e = hipMemcpyAsync(slot(2 * t + in), mine.src, mine.bytes, hipMemcpyDeviceToHost, stream_);
                    if (e == hipSuccess) e = hipEventRecord(events_[2 * t + in], stream_);
                }
                in ^= 1;
                const Piece& old = held[in];  // copied out while the new one is on its way
                if (e == hipSuccess && old.bytes) {
                    e = bounded_wait(watchdog_ms, [&] { return hipEventQuery(events_[2 * t + in]); });
                    if (e == hipSuccess) std::memcpy(old.dst, slot(2 * t + in), old.bytes);
                }
                if (e != hipSuccess) fault.store(static_cast<int>(e));
                if (!mine.bytes) return;
            }
        };
        std::vector<std::thread> helpers;
        try {
            helpers.reserve(n);
            for (uint32_t t = 1; t < n; t++) helpers.emplace_back(work, t);
        } catch (...) {  // no more threads: those there are take all pieces
        }
        work(0);
        for (std::thread& h : helpers) h.join();
        *err = static_cast<hipError_t>(fault.load());
        return *err == hipSuccess ? 0 : -1;
    }

    struct Piece {
        char* dst = nullptr;
        const char* src = nullptr;
        size_t bytes = 0;
    };

    char* slot(uint32_t k) const { return slots_ + k * kSlot; }

    // False while a call that failed may have left work that writes the slots.
    bool idle() {
        if (writing_ && hipStreamQuery(stream_) != hipErrorNotReady) writing_ = false;
        return !writing_;
    }

    bool reserve(uint32_t n) {
        if (n > n_slots_) {
            void* p = nullptr;
            if (hipHostMalloc(&p, n * kSlot, hipHostMallocDefault) != hipSuccess) {
                (void)hipGetLastError();
                return false;
            }
            if (slots_) (void)hipHostFree(slots_);
            slots_ = static_cast<char*>(p);
            n_slots_ = n;
        }
        while (events_.size() < n) {
            hipEvent_t e = nullptr;
            if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
                (void)hipGetLastError();
                return false;
            }
            events_.push_back(e);
        }
        return true;
    }

    // Without pinned memory: the runtime's own staging.
    template <class Ready>
    int direct(const std::vector<ReadPart>& parts, hipError_t* err, Ready&& ready) {
        int rc = ready();
        for (const ReadPart& p : parts) {
            if (rc || !p.bytes) continue;
            *err = hipMemcpyAsync(p.dst, p.src, p.bytes, hipMemcpyDeviceToHost, stream_);
            if (*err != hipSuccess) return -1;
        }
        return rc ? rc : ready();
    }

    int device_ = 0;
    hipStream_t stream_ = nullptr;
    bool writing_ = false;
    char* slots_ = nullptr;
    uint32_t n_slots_ = 0;
    std::vector<hipEvent_t> events_;
};

}  // namespace msim
