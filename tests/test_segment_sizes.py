"""Automatic segment sizes: the rule for the classic layouts and the sorted
state at the tables where it changes, and its bounds everywhere."""
import cxx
import pytest

PROGRAM = r"""
#include <cstdio>
#include "msim_host.hpp"
int main() {
    for (unsigned t = 12; t <= 28; t++)
        for (unsigned lw = 2; lw + 2 <= t; lw++) {
            std::printf("%u %u", t, lw);
            for (unsigned reach : {1u, 2u, 5u}) {
                std::printf(" %u %u", msim::auto_segment_log2(t, lw, reach, false),
                            msim::auto_segment_log2(t, lw, reach, true));
            }
            std::printf(" %u\n", msim::auto_sorted_segment_log2(t, lw));
        }
}
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    rows = [list(map(int, line.split())) for line in cxx.run(tmp_path_factory.mktemp("seg"), PROGRAM).splitlines()]
    return {(r[0], r[1]): r[2:] for r in rows}


def test_bounds(rule):
    for (t, lw), sizes in rule.items():
        assert all(9 <= s <= min(14, t) for s in sizes), (t, lw, sizes)
        assert all(s >= min(lw + 1, 14, t) for s in sizes), (t, lw, sizes)


@pytest.mark.parametrize("tlog,lw,reach,two_pass,look_back", [
    (13, 6, 2, 9, 9), (17, 8, 2, 10, 10), (19, 8, 2, 11, 11), (20, 10, 1, 11, 12), (20, 9, 2, 12, 12),
    (20, 5, 2, 9, 11), (21, 10, 1, 12, 12), (21, 9, 2, 13, 13), (22, 11, 1, 14, 14), (22, 9, 2, 13, 13),
    (23, 10, 2, 14, 14), (23, 12, 1, 14, 14), (24, 11, 2, 14, 14),
])
def test_classic_layouts(rule, tlog, lw, reach, two_pass, look_back):
    """Tables of 2^21 buckets and more need segments of many rows: in 4 rows a
    window is most of what a workgroup reads."""
    k = 2 * (reach - 1)
    assert rule[tlog, lw][k:k + 2] == [two_pass, look_back]


@pytest.mark.parametrize("tlog,lw,size", [(13, 6, 9), (17, 7, 10), (19, 8, 11), (21, 8, 11), (22, 9, 12), (24, 13, 14)])
def test_sorted_state(rule, tlog, lw, size):
    assert rule[tlog, lw][-1] == size
