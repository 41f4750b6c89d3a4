// msim_read.hpp — device-to-host readback through pinned slots that the
// handles of a device share, and the bounded wait the entry points share.
//
// A copy into the caller's (pageable) memory goes through the runtime's
// staging buffer, copied out by one thread which also takes
// the page faults of a fresh array: 64 MB of entities took 6.1 ms, 10 GB/s,
// where the link moves 56 GB/s (17 into pages that are there).  Here several
// threads each bring pieces into pinned slots of their own and copy them out,
// so link, copies and page faults overlap.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <memory>
#include <mutex>
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

// Waits for the work on a device's null stream, which a handle's non-blocking
// stream does not wait for.
inline hipError_t wait_null_stream(int device) {
    const DeviceScope scope(device);
    return hipStreamSynchronize(nullptr);
}

// The pinned slots of one device, lent to one readback at a time each and
// shared by the device's handles: 24 MB at most however many handles there
// are, given back to the system with the last of them.  Pinning costs about
// 70 us a MB, more than a readback of less than 30 MB gains by it, so the first
// one of those takes the runtime's path and only the second pins.  (Pinned by
// every handle in its first readback, a handle of 200k agents read once beside
// another took 2.3 ms where the runtime's path takes 1.0.)
class SlotPool {
public:
    // 64 MB of entities, two slots a thread, ms: slots of 0.5 MB 3.2 (every
    // transfer has a fixed cost), 1 MB 2.3, 2 MB 1.9, 4 MB 2.0; 4 threads 1.97,
    // 6 1.91, 8 1.94.
    static constexpr size_t kBytes = size_t{2} << 20;
    static constexpr uint32_t kMost = 12;
    static constexpr size_t kPinAtOnce = size_t{32} << 20;
    struct Slot {
        char* mem = nullptr;
        hipEvent_t done = nullptr;
    };
    struct Lease {
        Slot slot[kMost];
        uint32_t n = 0;
    };

    // The device's pool, for as long as someone holds it; null without memory
    // for it.
    static std::shared_ptr<SlotPool> of(int device) noexcept {
        static std::mutex m;
        static std::vector<std::weak_ptr<SlotPool>> pools;  // by device
        try {
            std::lock_guard<std::mutex> lk(m);
            const size_t d = static_cast<size_t>(std::max(device, 0));
            if (pools.size() <= d) pools.resize(d + 1);
            std::shared_ptr<SlotPool> p = pools[d].lock();
            if (!p) pools[d] = p = std::make_shared<SlotPool>(device);
            return p;
        } catch (...) {
            return nullptr;
        }
    }

    explicit SlotPool(int device) : device_(device) {}
    SlotPool(const SlotPool&) = delete;
    SlotPool& operator=(const SlotPool&) = delete;
    ~SlotPool() {  // nothing is lent: borrowers hold the pool
        const DeviceScope scope(device_);
        for (uint32_t k = 0; k < idle_.n; k++) (void)hipEventDestroy(idle_.slot[k].done);
        for (uint32_t k = 0; k < blocks_; k++) (void)hipHostFree(block_[k]);
    }

    // `least` to `want` slots for a readback of `bytes`, or none.
    void lend(Lease& to, uint32_t least, uint32_t want, size_t bytes) {
        std::lock_guard<std::mutex> lk(m_);
        const bool pin = used_ || bytes >= kPinAtOnce;
        used_ = true;
        const DeviceScope scope(device_);
        if (pin && idle_.n < want) grow(std::min(want - idle_.n, kMost - made_));
        to.n = 0;
        if (idle_.n < least) return;
        while (to.n < want && idle_.n > 0) to.slot[to.n++] = idle_.slot[--idle_.n];
    }

    void give_back(Lease& from) {
        std::lock_guard<std::mutex> lk(m_);
        while (from.n > 0) idle_.slot[idle_.n++] = from.slot[--from.n];
    }

private:
    // n more slots, in one allocation (12 of 2 MB each take 4 ms to free, one of
    // 24 MB 0.8); as many as there is memory and events for.
    void grow(uint32_t n) {
        void* p = nullptr;
        if (n == 0) return;
        if (hipHostMalloc(&p, n * kBytes, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            return;
        }
        block_[blocks_++] = p;
        made_ += n;
        for (uint32_t k = 0; k < n; k++) {
            Slot s{static_cast<char*>(p) + k * kBytes, nullptr};
            if (hipEventCreateWithFlags(&s.done, hipEventDisableTiming) != hipSuccess) {
                (void)hipGetLastError();
                return;
            }
            idle_.slot[idle_.n++] = s;
        }
    }

    const int device_;
    std::mutex m_;
    Lease idle_;
    void* block_[kMost] = {};
    uint32_t blocks_ = 0, made_ = 0;  // made_: slots in the blocks
    bool used_ = false;
};

class ReadBack {
public:
    // The handle's device and stream.
    void on(int device, hipStream_t stream) {
        device_ = device;
        stream_ = stream;
        pool_ = SlotPool::of(device);
    }

    static constexpr size_t kSlot = SlotPool::kBytes;

    // Pinned memory that kernels may write `bytes` of results to directly, for
    // the next read(); null past one slot, or when there is none to be had.  No
    // transfer follows the kernel.
    void* small(size_t bytes) {
        if (bytes > kSlot) return nullptr;
        refused_ = !borrow(1, 1, bytes);
        if (refused_) return nullptr;
        writing_ = true;
        return lease_.slot[0].mem;
    }
    static constexpr uint32_t kThreads = SlotPool::kMost / 2;

    ReadBack() = default;
    ReadBack(const ReadBack&) = delete;
    ReadBack& operator=(const ReadBack&) = delete;
    // The handle's stream has drained by now.
    ~ReadBack() {
        if (pool_) pool_->give_back(lease_);
    }

    // Reads the parts in stream order.  ready() waits for the stream (and
    // whatever else must hold before the caller's memory is written) and
    // returns 0, or a code that is passed on.  Otherwise returns 0, or -1 with
    // *err set (hipErrorNotReady: the watchdog expired).  After a failure the
    // slots stay with this handle, unused, until its stream has drained (idle).
    // host: the destinations are host memory, so nothing needs to be asked about
    // them for results of up to a slot (0.4 us each; a small state has six).
    template <class Ready>
    int read(const std::vector<ReadPart>& parts, uint32_t watchdog_ms, hipError_t* err, Ready&& ready,
             bool host = false) {
        const DeviceScope scope(device_);
        size_t total = 0;
        for (const ReadPart& p : parts) total += p.bytes;
        std::vector<ReadPart> known, rest;
        if (host && total <= kSlot) {
            rest = parts;
        } else {
            for (const ReadPart& p : parts) (by_runtime(p, total) ? known : rest).push_back(p);
        }
        int rc = rest.empty() && !known.empty() ? ready() : read_parts(rest, watchdog_ms, err, ready);
        if (rc == 0 && !known.empty()) rc = read_known(known, watchdog_ms, err);
        if (rc == 0) {
            writing_ = false;
        } else if (rc == -1 && *err != hipErrorNotReady) {
            (void)bounded_wait(watchdog_ms, [&] { return hipStreamQuery(stream_); });
        }
        if (idle() && pool_) pool_->give_back(lease_);
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
            there = there && lease_.n && p.src >= lease_.slot[0].mem && p.src < lease_.slot[0].mem + kSlot;
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
            if (refused_ || !borrow(1, 1, total)) {
                refused_ = false;
                return direct(parts, err, ready);
            }
            writing_ = true;
            char* const slot = lease_.slot[0].mem;
            size_t at = 0;
            for (const ReadPart& p : parts) {
                if (!p.bytes) continue;
                *err = hipMemcpyAsync(slot + at, p.src, p.bytes, hipMemcpyDeviceToHost, stream_);
                if (*err != hipSuccess) return -1;
                at += (p.bytes + 255) / 256 * 256;
            }
            const int rc = ready();
            if (rc) return rc;
            at = 0;
            for (const ReadPart& p : parts) {
                if (!p.bytes) continue;
                std::memcpy(p.dst, slot + at, p.bytes);
                at += (p.bytes + 255) / 256 * 256;
            }
            return 0;
        }
        // one thread per slot's worth, two slots each
        const uint32_t most = static_cast<uint32_t>(std::min<size_t>(kThreads, std::max<size_t>(1, total / kSlot)));
        if (!borrow(2, 2 * most, total)) return direct(parts, err, ready);
        const uint32_t n = lease_.n / 2;
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
                    const SlotPool::Slot& s = lease_.slot[2 * t + in];
                    e = hipMemcpyAsync(s.mem, mine.src, mine.bytes, hipMemcpyDeviceToHost, stream_);
                    if (e == hipSuccess) e = hipEventRecord(s.done, stream_);
                }
                in ^= 1;
                const Piece& old = held[in];  // copied out while the new one is on its way
                if (e == hipSuccess && old.bytes) {
                    const SlotPool::Slot& s = lease_.slot[2 * t + in];
                    e = bounded_wait(watchdog_ms, [&] { return hipEventQuery(s.done); });
                    if (e == hipSuccess) std::memcpy(old.dst, s.mem, old.bytes);
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

    // False while a call that failed may have left work that writes the slots.
    bool idle() {
        if (writing_ && hipStreamQuery(stream_) != hipErrorNotReady) writing_ = false;
        return !writing_;
    }

    // `least` to `want` slots in lease_.
    bool borrow(uint32_t least, uint32_t want, size_t bytes) {
        if (!pool_ || !idle()) return false;
        pool_->give_back(lease_);  // of a call that ended before its read()
        pool_->lend(lease_, least, want, bytes);
        return lease_.n != 0;
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
    bool refused_ = false;  // small() had no slot for the readback under way
    std::shared_ptr<SlotPool> pool_;
    SlotPool::Lease lease_;
};

}  // namespace msim
