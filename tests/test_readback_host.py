"""Readbacks on the host side (csrc/msim_read.hpp over a stand-in for the HIP
runtime): what cannot be brought about on one GPU, or only by breaking it."""
import os

import pytest

import cxx

FAKE = os.path.join(cxx.ROOT, "tests", "fake_hip")
PRELUDE = r"""
#include <cassert>
#include "msim_read.hpp"
using namespace msim;
constexpr size_t MB = size_t{1} << 20;
static std::vector<char> pattern(size_t bytes) {
    std::vector<char> v(bytes);
    for (size_t k = 0; k < bytes; k++) v[k] = static_cast<char>(k * 31 + k / 4093);
    return v;
}
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); std::exit(1); } } while (0)
"""


def check(tmp_path, body):
    assert cxx.run(tmp_path, PRELUDE + body, includes=[FAKE]) == "ok\n"


@pytest.mark.parametrize("megabytes", [1, 5, 40])
def test_another_device_is_current(tmp_path, megabytes):
    """The handle's device need not be the calling thread's, and the calling
    thread's stays what it was."""
    check(tmp_path, r"""
int main() {
    FakeStream stream;
    stream.device = 1;
    ReadBack rb;
    rb.on(1, &stream);
    const std::vector<char> src = pattern(%d * MB);
    std::vector<char> dst(src.size());
    hipError_t e = hipSuccess;
    CHECK(rb.read({{dst.data(), src.data(), src.size()}}, 1000, &e, [] { return 0; }) == 0);
    CHECK(e == hipSuccess && dst == src);
    CHECK(fake_device == 0);
    std::printf("ok\n");
}
""" % megabytes)


@pytest.mark.parametrize("megabytes", [1, 40])
def test_transfer_that_does_not_finish(tmp_path, megabytes):
    """A transfer past the watchdog is reported after the watchdog; the slots it
    may still write are neither used nor freed until the stream has drained."""
    check(tmp_path, r"""
int main() {
    FakeStream stream;
    ReadBack rb;
    rb.on(0, &stream);
    const std::vector<char> src = pattern(%d * MB);
    std::vector<char> dst(src.size());
    hipError_t e = hipSuccess;
    auto read = [&] {
        return rb.read({{dst.data(), src.data(), src.size()}}, 60, &e, [&] {
            return src.size() <= 2 * MB && stream.stuck ? 5 : 0;  // small ones: what waits is ready()
        });
    };
    CHECK(read() == 0 && dst == src);
    stream.stuck = true;
    const auto t0 = std::chrono::steady_clock::now();
    const int rc = read();
    CHECK(rc == 5 || (rc == -1 && e == hipErrorNotReady));
    CHECK(std::chrono::steady_clock::now() - t0 < std::chrono::milliseconds(1000));
    CHECK(fake().unbounded_waits == 0);
    const int frees = fake().frees;
    CHECK(rb.small(100) == nullptr);
    CHECK(fake().frees == frees);
    stream.stuck = false;
    dst.assign(dst.size(), 0);
    CHECK(rb.small(100) != nullptr);
    CHECK(read() == 0 && dst == src);
    std::printf("ok\n");
}
""" % megabytes)


@pytest.mark.parametrize("kilobytes", [3, 1000, 5000, 40000])
def test_destinations_the_runtime_knows(tmp_path, kilobytes):
    """Device memory is never written by the host; pinned memory takes one copy
    where the results do not fit a slot; both beside ordinary memory."""
    check(tmp_path, r"""
#include <sys/mman.h>
int main() {
    FakeStream stream;
    ReadBack rb;
    rb.on(0, &stream);
    const size_t bytes = size_t{1000} * %d;
    const std::vector<char> src = pattern(3 * bytes);
    std::vector<char> pageable(bytes), own(bytes);
    char* device = static_cast<char*>(mmap(nullptr, bytes, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0));
    fake().on_device[device] = bytes;
    fake().pinned[own.data()] = own.size();
    hipError_t e = hipSuccess;
    auto is = [&](const std::vector<char>& v, size_t from) { return std::memcmp(v.data(), src.data() + from, bytes) == 0; };
    CHECK(rb.read({{device, src.data(), bytes}, {pageable.data(), src.data() + bytes, bytes},
                   {own.data(), src.data() + 2 * bytes, bytes}}, 1000, &e, [] { return 0; }) == 0);
    CHECK(fake().copied_to[device] == bytes);
    CHECK(is(pageable, bytes) && is(own, 2 * bytes));
    if (3 * bytes > 2 * MB) CHECK(fake().copied_to[own.data()] == bytes);
    // what a kernel has written to a slot
    if (void* slot = rb.small(1000)) {
        std::memcpy(slot, src.data(), 1000);
        fake().copied_to.clear();
        CHECK(rb.read({{device, slot, 1000}}, 1000, &e, [] { return 0; }) == 0);
        CHECK(fake().copied_to[device] == 1000);
    }
    std::printf("ok\n");
}
""" % kilobytes)


def test_slots_are_shared_bounded_and_given_back(tmp_path):
    """The first readback of a few megabytes does not pin, the second does, a
    large one at once; 64 handles pin no more than one, and the last one gives
    everything back."""
    check(tmp_path, r"""
static void read(ReadBack& rb, size_t bytes) {
    const std::vector<char> src = pattern(bytes);
    std::vector<char> dst(bytes);
    hipError_t e = hipSuccess;
    CHECK(rb.read({{dst.data(), src.data(), bytes}}, 1000, &e, [] { return 0; }) == 0 && dst == src);
}
static void read_written(ReadBack& rb, size_t bytes) {  // by a kernel, to a slot if there is one
    const std::vector<char> src = pattern(bytes);
    std::vector<char> stage(bytes), dst(bytes);
    char* to = static_cast<char*>(rb.small(bytes));
    if (!to) to = stage.data();
    std::memcpy(to, src.data(), bytes);
    hipError_t e = hipSuccess;
    CHECK(rb.read({{dst.data(), to, bytes}}, 1000, &e, [] { return 0; }) == 0 && dst == src);
}
int main() {
    FakeStream stream;
    for (int large = 0; large < 3; large++) {
        ReadBack rb;
        rb.on(0, &stream);
        const int pins = fake().pins;
        const size_t bytes = large == 2 ? 40 * MB : (large ? 5 * MB : 1 * MB);
        if (large) read(rb, bytes); else read_written(rb, bytes);
        CHECK((fake().pins != pins) == (large == 2));
        if (large) read(rb, bytes); else read_written(rb, bytes);
        CHECK(fake().pinned_bytes == (large == 2 ? 24 : (large ? 8 : 2)) * MB);
        read(rb, bytes);
        CHECK(fake().pins == pins + 1);
    }
    CHECK(fake().pinned_bytes == 0);
    {
        std::vector<std::unique_ptr<ReadBack>> all;
        for (int k = 0; k < 64; k++) {
            all.emplace_back(new ReadBack);
            all.back()->on(k % 2, &stream);
            stream.device = k % 2;
            read(*all.back(), 33 * MB);
            read_written(*all.back(), MB);
        }
        CHECK(fake().pinned_bytes == 2 * 24 * MB);  // two devices
        const int frees = fake().frees;
        all.resize(2);
        CHECK(fake().frees == frees);
    }
    CHECK(fake().pinned_bytes == 0);
    fake().no_pinning = true;
    ReadBack rb;
    rb.on(0, &stream);
    for (int k = 0; k < 3; k++) {
        read(rb, 40 * MB);
        read(rb, MB);
        read_written(rb, MB);
    }
    std::printf("ok\n");
}
""")


def test_readers_in_several_threads(tmp_path):
    check(tmp_path, r"""
int main() {
    std::vector<std::thread> threads;
    const std::vector<char> src = pattern(20 * MB);
    std::atomic<int> wrong{0};
    for (int t = 0; t < 4; t++) {
        threads.emplace_back([&, t] {
            FakeStream stream;
            std::vector<char> dst(src.size());
            for (int round = 0; round < 3; round++) {
                ReadBack rb;
                rb.on(0, &stream);
                for (int k = 0; k < 12; k++) {
                    const size_t bytes = k %% 3 == 0 ? 1000 + 7 * t : (k %% 3 == 1 ? 3 * MB + t : src.size() - t);
                    std::memset(dst.data(), 0, bytes);
                    char* to = static_cast<char*>(rb.small(bytes));
                    if (to) std::memcpy(to, src.data() + t, bytes - t);
                    hipError_t e = hipSuccess;
                    const int rc = rb.read({{dst.data(), to ? to : src.data() + t, bytes - t}}, 1000, &e, [] { return 0; });
                    if (rc != 0 || std::memcmp(dst.data(), src.data() + t, bytes - t) != 0) wrong++;
                    if (fake().pinned_bytes > 24 * MB) wrong++;
                }
            }
        });
    }
    for (std::thread& t : threads) t.join();
    CHECK(wrong == 0);
    CHECK(fake().pinned_bytes == 0);
    std::printf("ok\n");
}
""".replace("%%", "%"))


def test_slots_of_a_stuck_handle_are_not_lent(tmp_path):
    """What a stuck handle's work may still write stays with it until its stream
    has drained."""
    check(tmp_path, r"""
int main() {
    FakeStream good, bad;
    const std::vector<char> src = pattern(10 * MB);
    std::vector<char> dst(src.size());
    hipError_t e = hipSuccess;
    ReadBack other;
    other.on(0, &good);
    auto fine = [&](size_t bytes) {
        std::memset(dst.data(), 0, bytes);
        CHECK(other.read({{dst.data(), src.data(), bytes}}, 100, &e, [] { return 0; }) == 0);
        CHECK(std::memcmp(dst.data(), src.data(), bytes) == 0);
    };
    fine(MB);
    fine(MB);
    {
        ReadBack rb;
        rb.on(0, &bad);
        void* mine = rb.small(1000);
        CHECK(mine);
        bad.stuck = true;
        std::vector<char> out(1000);
        CHECK(rb.read({{out.data(), mine, 1000}}, 20, &e, [] { return 5; }) == 5);
        for (int k = 0; k < 3; k++) fine(MB);
        for (int k = 0; k < 3; k++) fine(10 * MB);
        for (int k = 0; k < 20; k++) {
            void* s = other.small(10);
            CHECK(s != mine);
            CHECK(other.read({{dst.data(), s ? s : src.data(), 10}}, 100, &e, [] { return 0; }) == 0);
        }
        CHECK(fake().frees == 0);
        bad.stuck = false;
        std::memset(mine, 7, 1000);
        CHECK(rb.read({{out.data(), src.data(), 1000}}, 20, &e, [] { return 0; }) == 0);
        CHECK(std::memcmp(out.data(), src.data(), 1000) == 0);
    }
    std::printf("ok\n");
}
""")


def test_null_stream_of_the_handles_device(tmp_path):
    """A handle's parameters may come from the null stream of its device, which
    need not be the current one."""
    check(tmp_path, r"""
int main() {
    for (int current = 0; current < 2; current++) {
        hipSetDevice(current);
        CHECK(wait_null_stream(1) == hipSuccess);
        CHECK(fake().null_stream_device == 1 && fake_device == current);
    }
    std::printf("ok\n");
}
""")
