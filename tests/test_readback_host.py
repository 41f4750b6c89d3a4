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
    const bool direct = 3 * bytes > 2 * MB;
    CHECK(fake().copied_to.count(own.data()) == (direct ? 1u : 0u));
    if (direct) CHECK(fake().copied_to[own.data()] == bytes);
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
