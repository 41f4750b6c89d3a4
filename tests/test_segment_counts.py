"""Layout of the sums over groups of segments: few words to add up before any
segment, few sums in one cache line for the workgroups to meet on."""
import cxx

PROGRAM = r"""
#include <cstdio>
#include "msim_host.hpp"
int main() {
    for (unsigned l = 0; l <= 19; l++) {
        for (unsigned n : {(1u << l) - (l > 0), 1u << l, (1u << l) + 1u}) {
            std::printf("%u %u %u %u\n", n, msim::seg_group_log2(n), msim::kGroupStride, msim::seg_group_words(n));
        }
    }
}
"""


def test_groups_of_segments(tmp_path):
    rows = [tuple(map(int, line.split())) for line in cxx.run(tmp_path, PROGRAM).splitlines()]
    assert len(rows) == 60
    for n, log, stride, words in rows:
        groups = (n - 1 >> log) + 1
        assert words >= (groups - 1) * stride + 1, f"{n} segments: no word for the last group"
        assert 128 // (4 * stride) * 2 ** log <= max(64, 4 * 2 ** log), f"{n} segments: sums too close together"
        # words a workgroup adds up: the groups before its own, the segments before it in its group
        assert groups - 1 + 2 ** log - 1 <= max(31, 3 * n ** 0.5), f"{n} segments"
