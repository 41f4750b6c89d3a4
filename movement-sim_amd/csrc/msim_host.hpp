// msim_host.hpp — host-side helpers shared by the C-ABI entry points:
// map/agent validation, grid sizing and the exact squared-radius threshold.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <string>

#include "msim/types.h"

namespace msim {

inline uint32_t next_pow2_u32(uint32_t v) {
    if (v <= 1) return 1;
    v--;
    v |= v >> 1;
    v |= v >> 2;
    v |= v >> 4;
    v |= v >> 8;
    v |= v >> 16;
    return v + 1;
}

inline uint32_t ceil_log2_u64(uint64_t v) {
    uint32_t l = 0;
    while ((1ull << l) < v) l++;
    return l;
}

// Bucket table size: about one bucket per agent, at least 2^12 (one scan
// tile) and at most 2^26.
inline uint32_t auto_table_log2(uint32_t n_agents) {
    uint32_t l = ceil_log2_u64(n_agents ? n_agents : 1);
    if (l < 12) l = 12;
    if (l > 26) l = 26;
    return l;
}

// Table rows: the table must fold the world vertically (height <= the
// world's rows in cells), otherwise rows the world never reaches stay empty
// and the used buckets alias more.  Beyond that, rows are kept narrow so the
// rebinning window (a segment plus a few rows each side) stays small.
inline uint32_t auto_width_log2(uint32_t tlog, uint32_t rows_log) {
    uint32_t fold = rows_log + 2 > tlog ? 2 : tlog - rows_log;  // height <= 2^rows_log
    uint32_t l = fold < 5 ? 5 : fold;
    if (l + 2 > tlog) l = tlog - 2;
    return l;
}

// Segment sizes: two table rows at least (a window adds reach + 1 rows on
// both sides), up to 2^14 buckets (64 KB of LDS counters).
inline uint32_t segment_in_bounds(uint32_t l, uint32_t tlog, uint32_t lw) {
    if (l < lw + 1u) l = lw + 1u;
    if (l > 14) l = 14;
    return l > tlog ? tlog : l;
}

// Segment owned by one rebinning workgroup of the classic layouts (reach:
// cells an agent moves at most in a tick, plus one; look_back: binning 2):
// 16 table rows, against which the rows a window adds are few, but of small
// tables about 128 segments, so that the CUs have work; where a window adds
// two rows a side (reach 1) fewer rows do.  Ticks, us:
//   two passes, reach 1: 2^22 buckets in rows of 2^11, 2.2M agents, 116 at
//     2^14, 127 at 2^13, 133 at 2^12; 2^21, rows of 2^10, 1.1M agents, 79, 71,
//     66 and 70 at 2^11; 2^20, rows of 2^10, 1M agents, 115, 104, 85, 81;
//   reach 2: 2^23, rows of 2^10, 4.3M agents, 233, 248, 263; 2^21, rows of
//     2^9, 2M agents, 120, 105, 109, 132; 2^20, rows of 2^9, 1M agents, 88,
//     69, 61, 72; 2^20, rows of 2^5, 94 at 2^12, 73 at 2^11, 63 at 2^9;
//     123k agents on 2^17, 39 at 2^12, 34 at 2^11, 33 at 2^10 and 2^9;
//   look-back: 2^23, rows of 2^10, 216 at 2^14, 235 at 2^12; 2^20, rows of
//     2^9, reach 1, 61 at 2^12, 64 at 2^11; 2^19, rows of 2^6, 300k agents, 38
//     at 2^11, 44 at 2^10.
inline uint32_t auto_segment_log2(uint32_t tlog, uint32_t lw, uint32_t reach, bool look_back) {
    uint32_t most = 9;
    if (tlog >= 22u) most = 14;
    else if (tlog == 21u) most = reach < 2u ? 12u : 14u;
    else if (tlog == 20u) most = reach < 2u && !look_back ? 11u : 12u;
    else if (tlog > 16u) most = tlog > 18u ? 11u : tlog - 7u;
    // a look-back chain of many small segments is slow
    const uint32_t least = tlog > 20u ? 10u : (look_back ? (most < 11u ? most : 11u) : 9u);
    uint32_t l = lw + 4u;
    if (l > most) l = most;
    if (l < least) l = least;
    return segment_in_bounds(l, tlog, lw);
}

// The same for the sorted state: about 128 segments of 2^9 to 2^11 buckets
// (2^12 in tables of 2^22 and more).  Ticks of 1.6M agents on 2^21 buckets in
// rows of 2^8, us: 89 at 2^14, 62 at 2^13, 61 at 2^12 and 2^11, 72 at 2^10; 9M
// on 2^24 in rows of 2^11: 433, 341, 348, 432, 1,199; 300k on 2^19 in rows of
// 2^8: 66, 40, 28, 24, 28.
inline uint32_t auto_sorted_segment_log2(uint32_t tlog, uint32_t lw) {
    return segment_in_bounds(tlog > 21u ? 12u : (tlog > 18u ? 11u : (tlog > 16u ? tlog - 7u : 9u)), tlog, lw);
}

// The same for one of many tables in a launch, of `buckets` in all, whose
// segments fill the GPU together: 2^11 buckets, fewer while that leaves less
// than 384 segments.  Count + place of 64 scenarios of 5.8M agents: 210 us at
// 2^9 buckets (16 rows), 127 at 2^10, 92 at 2^11 and 2^12, 118 at 2^13; a
// differentiable run of 7 scenarios on 2^16 buckets each was 2% slower at 2^11
// (224 segments) than at 2^10.
inline uint32_t auto_batch_segment_log2(uint64_t buckets, uint32_t tlog, uint32_t lw) {
    uint32_t l = 11;
    while (l > 9 && (buckets >> l) < 384u) l--;
    return segment_in_bounds(l, tlog, lw);
}

// Cells an agent of at most this speed moves per axis and tick at most, plus
// one (the heading has |dir| = speed up to rounding).
inline uint32_t cell_reach(float max_speed, float cell) {
    return static_cast<uint32_t>(std::floor(max_speed * (1.0f + 1.0f / 1048576.0f) / cell)) + 1u;
}

// Window slots each rebinning thread loads per round.  Segments of up to 2^11
// buckets have windows of at most about 4,000 slots, which 512 threads with 8
// each load mostly past the end: ticks of 10k agents 28.0 us with 8, 26.0 with
// 4; 123k 30.8, 28.8; 1M 53.4, 51.0; 16 scenarios 34.6, 31.4.  At 2^12 buckets
// (8M agents) 8 keep more loads in flight: 414 us, 431 with 4.  Segments of
// 2^14 buckets (64 KB of LDS counters, two workgroups per CU) measured faster
// with 4.
inline uint32_t auto_bin_unroll(uint32_t seg_log) { return seg_log == 12u || seg_log == 13u ? 8u : 4u; }

// Sums of the sorted state's per-segment counts, over groups of 2^l
// consecutive segments: every move workgroup adds up the groups before its own
// segment's and the segments before it in its group, so l is about half of
// log2(n_seg) (at least 4) and neither has more than about sqrt(n_seg) words
// (2^17 segments: 512 + 255; groups of 16 would be 8,192).
constexpr uint32_t seg_group_log2(uint32_t n_seg) {
    uint32_t l = 0;
    while (l < 31u && (1u << l) < n_seg) l++;
    return l > 8u ? l / 2u : 4u;
}
// Words from one group's sum to the next.  Side by side, 32 sums share a cache
// line, to which every workgroup then adds: see SegCounts.
constexpr uint32_t kGroupStride = 8;
constexpr uint32_t seg_group_words(uint32_t n_seg) {
    return ((n_seg + (1u << seg_group_log2(n_seg)) - 1u) >> seg_group_log2(n_seg)) * kGroupStride;
}

// Bounding box of the roads and agents.
struct Extent {
    float x0 = 0.0f, x1 = 0.0f, y0 = 0.0f, y1 = 0.0f;
    // Cells spanned (one past the last).
    double cols(float cell) const { return std::floor(double{x1} / cell) - std::floor(double{x0} / cell) + 1.0; }
    double rows(float cell) const { return std::floor(double{y1} / cell) - std::floor(double{y0} / cell) + 1.0; }
};

inline Extent extent_of(const msim_road* roads, uint32_t n_roads, const msim_entity* e, uint32_t n) {
    Extent b;
    auto add = [&](float x, float y) {
        b.x0 = std::min(b.x0, x);
        b.x1 = std::max(b.x1, x);
        b.y0 = std::min(b.y0, y);
        b.y1 = std::max(b.y1, y);
    };
    if (n_roads) {
        b = Extent{roads[0].start.pos.x, roads[0].start.pos.x, roads[0].start.pos.y, roads[0].start.pos.y};
    } else if (n) {
        b = Extent{e[0].pos.x, e[0].pos.x, e[0].pos.y, e[0].pos.y};
    }
    for (uint32_t r = 0; r < n_roads; r++) {
        add(roads[r].start.pos.x, roads[r].start.pos.y);
        add(roads[r].end.pos.x, roads[r].end.pos.y);
    }
    for (uint32_t i = 0; i < n; i++) {
        add(e[i].pos.x, e[i].pos.y);
    }
    return b;
}

// floor(log2(rows spanned, in cells)), at least 2.
inline uint32_t extent_rows_log2(const Extent& b, float cell) {
    const double rows = (double{b.y1} - double{b.y0}) / cell + 1.0;
    uint32_t l = 2;
    while (l < 30 && static_cast<double>(1ull << (l + 1)) <= rows) l++;
    return l;
}

// A table that holds the whole world, one bucket per cell, where that takes
// no more buckets than the agents' own table (2^tlog): its rows are as short
// as the world, so the rebinning windows are narrow, and no bucket mixes far
// cells.  (Folded onto rows of 2^11, 1M agents in a world of 781 x 781 cells
// had 62% of each row empty.)  Crowded worlds gain too, although few segments
// hold all their agents, since the neighbour pass is most of their ticks: 70k
// agents on 17 x 17 cells take 545 us on 2^12 buckets, where one segment has
// 65k of them, and 620 on their own 2^17.  Past 8,192 agents per 512 buckets
// the agents' own table stays.
inline bool whole_world_table(uint32_t n, double rows, double cols, uint32_t* tlog, uint32_t* lw) {
    auto ceil_log2 = [](double v) {
        uint32_t l = 0;
        while (l < 31 && static_cast<double>(1ull << l) < v) l++;
        return l;
    };
    const uint32_t cr = std::max(2u, ceil_log2(rows)), cc = std::max(2u, ceil_log2(cols));
    const uint32_t t = std::max(12u, cr + cc);
    if (t > *tlog || (static_cast<uint64_t>(n) >> 13) > (1ull << (t - 9u))) return false;
    *tlog = t;
    *lw = cc;
    return true;
}

// Ticks per captured segment: whole reorder periods (at least one), about
// graph_ticks long; graph_ticks itself when reordering is off.
inline uint32_t segment_ticks(uint32_t graph_ticks, uint32_t reorder_interval) {
    if (reorder_interval == 0) return graph_ticks;
    uint32_t k = (graph_ticks + reorder_interval / 2) / reorder_interval;
    if (k == 0) k = 1;
    return k * reorder_interval;
}

inline bool is_pow2_float(float v) {
    if (!(v > 0.0f) || !std::isfinite(v)) return false;
    int e = 0;
    return std::frexp(v, &e) == 0.5f;
}

// Smallest power of two >= r: with such a cell edge, floor(x / cell) is exact
// and any two points closer than r lie in the same or adjacent cells.
inline float pow2_cell(float r) {
    int e = 0;
    const float m = std::frexp(r, &e);
    if (m == 0.5f) return r;
    return std::ldexp(1.0f, e);
}

inline float bits_to_float(uint32_t b) {
    float f;
    std::memcpy(&f, &b, 4);
    return f;
}

// Smallest binary32 x >= 0 with sqrtf(x) >= r.  sqrtf is correctly rounded
// and non-decreasing, so sqrtf(d2) < r  <=>  d2 < d2_limit_for(r).
inline float d2_limit_for(float r) {
    uint32_t lo = 0, hi = 0x7f800000u;  // +inf
    while (lo < hi) {
        const uint32_t mid = lo + (hi - lo) / 2;
        volatile float x = bits_to_float(mid);
        if (std::sqrt(static_cast<float>(x)) >= r) {
            hi = mid;
        } else {
            lo = mid + 1;
        }
    }
    return bits_to_float(lo);
}

// The neighbour predicate drops quad_tree_in_range's box tests, which is exact
// when every |dx| > r already fails d2 < limit, i.e. when fl(r*r) >= limit.
inline bool box_tests_implied(float r, float limit) {
    volatile float rr = r;
    const float sq = rr * rr;
    return sq >= limit;
}

// Every read random_move.comp:778-828 can make must stay inside the arrays:
// an endpoint with count >= 3 may read connections[index + count] (the draw
// can return the top offset), count == 2 reads connections[index + 1].
inline bool validate_map(const msim_road* roads, uint32_t n_roads, const uint32_t* conns,
                         uint32_t n_conns, std::string* why) {
    char buf[256];
    for (uint32_t r = 0; r < n_roads; r++) {
        const msim_coordinate* ends[2] = {&roads[r].start, &roads[r].end};
        for (int k = 0; k < 2; k++) {
            const msim_coordinate& c = *ends[k];
            if (!std::isfinite(c.pos.x) || !std::isfinite(c.pos.y)) {
                snprintf(buf, sizeof(buf), "road %u has a non-finite endpoint", r);
                *why = buf;
                return false;
            }
            if (c.connectedCount >= (1u << 24)) {
                // float(count) must be exact for the draw to stay <= count
                snprintf(buf, sizeof(buf), "road %u %s group count %u exceeds 2^24", r,
                         k ? "end" : "start", c.connectedCount);
                *why = buf;
                return false;
            }
            uint64_t top = 0;
            if (c.connectedCount == 2) {
                top = static_cast<uint64_t>(c.connectedIndex) + 1;
            } else if (c.connectedCount >= 3) {
                top = static_cast<uint64_t>(c.connectedIndex) + c.connectedCount;
            } else {
                continue;
            }
            if (top >= n_conns) {
                snprintf(buf, sizeof(buf),
                         "road %u %s group (index %u, count %u) can read connections[%llu] but only "
                         "%u entries exist; append a guard entry",
                         r, k ? "end" : "start", c.connectedIndex, c.connectedCount,
                         static_cast<unsigned long long>(top), n_conns);
                *why = buf;
                return false;
            }
        }
    }
    for (uint32_t k = 0; k < n_conns; k++) {
        if (conns[k] >= n_roads) {
            snprintf(buf, sizeof(buf), "connections[%u] = %u is not a road index (< %u)", k, conns[k],
                     n_roads);
            *why = buf;
            return false;
        }
    }
    return true;
}

// Cell coordinates must stay far from the +-2^30 clamp of the cell index so
// that every tick's displacement bound holds in cell units.
inline bool validate_extent(const msim_road* roads, uint32_t n_roads, const msim_entity* e, uint32_t n,
                            float inv_cell, std::string* why) {
    const double lim = 536870912.0;  // 2^29 cells
    auto bad = [&](float v) { return !(std::fabs(static_cast<double>(v) * inv_cell) < lim); };
    char buf[160];
    for (uint32_t r = 0; r < n_roads; r++) {
        if (bad(roads[r].start.pos.x) || bad(roads[r].start.pos.y) || bad(roads[r].end.pos.x) ||
            bad(roads[r].end.pos.y)) {
            snprintf(buf, sizeof(buf), "road %u lies beyond 2^29 grid cells from the origin", r);
            *why = buf;
            return false;
        }
    }
    for (uint32_t i = 0; i < n; i++) {
        if (bad(e[i].pos.x) || bad(e[i].pos.y) || bad(e[i].target.x) || bad(e[i].target.y)) {
            snprintf(buf, sizeof(buf), "agent %u lies beyond 2^29 grid cells from the origin", i);
            *why = buf;
            return false;
        }
    }
    return true;
}

inline bool validate_entities(const msim_entity* e, uint32_t n, uint32_t n_roads, const float* speed,
                              std::string* why) {
    char buf[256];
    for (uint32_t i = 0; i < n; i++) {
        if (e[i].roadIndex >= n_roads) {
            snprintf(buf, sizeof(buf), "agent %u has roadIndex %u >= %u roads", i, e[i].roadIndex, n_roads);
            *why = buf;
            return false;
        }
        if (!std::isfinite(e[i].pos.x) || !std::isfinite(e[i].pos.y) || !std::isfinite(e[i].target.x) ||
            !std::isfinite(e[i].target.y)) {
            snprintf(buf, sizeof(buf), "agent %u has a non-finite position or target", i);
            *why = buf;
            return false;
        }
        if (speed && !(speed[i] >= 0.0f && std::isfinite(speed[i]))) {
            snprintf(buf, sizeof(buf), "agent %u has an invalid speed", i);
            *why = buf;
            return false;
        }
    }
    return true;
}

}  // namespace msim
