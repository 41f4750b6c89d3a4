// msim_sorted.hpp — the move dispatch on bucket-sorted agent state.
//
// The hot agent state (position; target, speed and caller index in one
// 16-byte record) is kept in the slot order of the current binning, so the
// binning needs no slot -> agent map and positions need no gather.  One launch per move dispatch advances
// every agent (random_move.comp:830-852) and writes it, together with the
// rest of its hot state, straight into the next binning's slot order:
//
//   * the toroidal bucket table is cut into segments; workgroup `seg` owns
//     the slots of the agents whose new bucket lies in its segment (segments
//     dealt to the XCDs in runs, so that neighbouring windows share an L2);
//   * every slot carries `nxt`, the bucket of its agent's next position,
//     computed when the agent was last placed; counting and ranking read
//     these 4 bytes per slot and no state;
//   * an agent moves at most D cells per axis, so it lands within `margin`
//     buckets of its previous bucket.  With lists (LISTS), whoever placed an agent that will leave its segment also
//     listed it (slot, next bucket) for the segment above or below: the
//     segment's agents are among its own previous slots and its two
//     neighbours' lists.  Otherwise they are sought in a window of the
//     previous slot order, the segment and the margin on both sides;
//   * the segment's first slot follows from counts made before the launch:
//     the previous move and route choice counted, per segment and per group
//     of segments (SegCounts), the agents whose next bucket lies in it, so no
//     segment waits for another.  Inside run_ticks every workgroup sums the
//     counts before its segment itself; a single dispatch runs k_seg_scan
//     first;
//   * rank: the window entries whose `nxt` lies in the segment take their new
//     slots from LDS counters; an LDS map records, per new slot, the old
//     slot's window index and the counted bucket;
//   * store pass: the new slots in order (whole lines written per wave),
//     each agent's position and record gathered from its old slot through
//     the map, moved, checked against its counted bucket and stored with the
//     bucket of its following move as the new `nxt`;
//   * arrivals are stored at once but for what the route choice decides
//     (target, next bucket, heading): each is listed (new slot, caller index,
//     position, speed) in the segment's own slice [base, base + total) of
//     the arrival list, and k_route_sorted, launched next, routes every
//     segment's list (random_move.comp:778-828).  Road and PRNG state live in
//     caller order, 32 bytes per agent with the connection index and count
//     of the endpoint the agent heads to, and are touched only there.
//
// Each agent's arithmetic is the plain tick's exactly; only where the state
// is stored changes.  The agents' order inside a bucket follows the rank
// pass's LDS atomics and carries no meaning: no result depends on it.
#pragma once

#include "msim_bin.hpp"
#include "msim_host.hpp"

namespace msim {

// pos + heading of an agent that keeps walking (random_move.comp:830-846).
// The sorted move evaluates it twice for every agent and tick: for the move
// itself and, one tick earlier, to bin the agent's next position.  Both must
// round alike.  With contraction on, the compiler may fuse p + d differently
// at different call sites, so that build keeps a single out-of-line copy.
#ifdef MSIM_CONTRACTED
#define MSIM_WALK_ATTR __device__ __noinline__
#else
#define MSIM_WALK_ATTR __device__ __forceinline__
#endif
MSIM_WALK_ATTR float4 walk_step(float px, float py, float dx, float dy, float len, float s) {
    const float hx = (dx / len) * s;
    const float hy = (dy / len) * s;
    return make_float4(px + hx, py + hy, hx, hy);
}

// Position after the next move from p toward t at speed s: the step, or the
// target itself on arrival (random_move.comp:841-852).
__device__ __forceinline__ float2 next_position(float2 p, float2 t, float s) {
    const float dx = t.x - p.x;
    const float dy = t.y - p.y;
    const float len = vlen(dx, dy);
    if (len > s) {
        const float4 w = walk_step(p.x, p.y, dx, dy, len, s);
        return make_float2(w.x, w.y);
    }
    return t;
}

// Hot agent state in slot order (one copy per binning buffer).  Target,
// speed and caller index share one 16-byte record, so that moving an agent
// takes two gathers (position, record) and three stores (position, record,
// next bucket): a scattered gather costs about the same per instruction
// whatever its width, so fewer, wider ones are cheaper.  Positions and next
// buckets stay separate arrays, which the neighbour pass and the count
// passes stream alone.
struct SortedBufs {
    float2* pos;    // [n + pad]
    uint4* rec;     // [n] {target x, target y, speed (float bits; unused with spd_const), caller index}
    uint32_t* nxt;  // [n] bucket (in the agent's table) of its next position
    float2* dir;    // [n + pad] heading, written on a batch's last tick only
};

__device__ __forceinline__ uint4 hot_record(float2 tgt, float spd, uint32_t caller) {
    return make_uint4(__float_as_uint(tgt.x), __float_as_uint(tgt.y), __float_as_uint(spd), caller);
}

// Caller-order route state of one agent (cold[2 h], cold[2 h + 1]): road,
// connection index and count of the endpoint it heads to (route_endpoint),
// and the PRNG state.
__device__ __forceinline__ uint4 cold_word(uint32_t road, uint2 c) { return make_uint4(road, c.x, c.y, 0u); }

// Agents whose next bucket lies in each segment, and the sums of those
// counts over groups of 2^log consecutive segments (seg_group_log2): a
// segment's first slot is then the sum of the groups before its own and of the
// segments before it in its group, which the workgroup of the segment adds up
// while its window is in flight.
// The groups' words are bound by the atomics that meet in one cache line, some
// 6 ns each: a workgroup adds to its segment and its neighbours, which are
// mostly of one group, so it adds their sum at once (leave_flush, next_flush),
// and the words lie kGroupStride apart.  Ticks of 1M agents, us, each count
// added to its group by itself and the words side by side -> as here: 512
// segments 48 -> 41, 1,024 66 -> 48, 2,048 84 -> 64; 100k agents on 256
// segments 39 -> 22; without the sums over groups at all 40, 47, 63, 21.
struct SegCounts {
    uint32_t* seg;    // [n_seg]
    uint32_t* group;  // [seg_group_words(n_seg)]
    uint32_t log;
    __device__ void add_seg(uint32_t g, uint32_t v) const { atomicAdd(&seg[g], v); }
    __device__ void add_group(uint32_t gg, uint32_t v) const { atomicAdd(&group[gg * kGroupStride], v); }
    __device__ void add(uint32_t g, uint32_t v) const {
        add_seg(g, v);
        add_group(g >> log, v);
    }
    __device__ void clear(uint32_t g) const {
        seg[g] = 0u;
        if ((g & ((1u << log) - 1u)) == 0u) group[(g >> log) * kGroupStride] = 0u;
    }
    // Thread tid's part of the counts before segment g (summed over the
    // workgroup's threads).
    __device__ uint32_t before(uint32_t g, uint32_t tid, uint32_t threads) const {
        const uint32_t gg = g >> log;
        uint32_t v = 0;
        for (uint32_t k = tid; k < gg; k += threads) v += group[k * kGroupStride];
        for (uint32_t k = (gg << log) + tid; k < g; k += threads) v += seg[k];
        return v;
    }
};

// What one segment hands to the next move (LISTS): its slots [x, y) and the
// lengths of its two lists of agents whose next bucket lies in another
// segment.  Both lists use the segment's own range of the list array, an
// entry {slot, next bucket} for each: the z agents going to the segment
// above from the front, the w agents going below from the back.  An agent is
// listed at most once, so the range holds them all.  "Above" and "below" are
// cyclic in the table; with two segments everything goes above.
struct SegLists {
    uint4* rec;    // [n_seg]
    uint2* leave;  // [n]
};

struct SortedMove {
    SortedBufs src, dst;
    SegLists from, to;   // LISTS: the lists this move reads, and those it and the route choice write
    uint4* arr_rec;      // [n] arrivals {new slot, caller index, x bits, y bits}, segment g's at
                         // [seg_start[g], + seg_arr[g])
    float* arr_spd;      // [n] their speeds; nullptr with spd_const
    uint32_t* seg_start;        // [n_seg + 1] first slot of each segment (k_seg_scan, or written by the move)
    SegCounts cur;              // counts this move consumes (cur.seg nullptr: k_seg_scan did)
    SegCounts next;             // counts for the next move
    uint32_t* seg_arr;          // [n_seg] arrivals of each segment
    uint4* cold;                // [2 n] caller order: cold_word, PRNG state
    uint32_t n;
    const msim_road* roads;
    const uint32_t* conns;
    float spd_const;
    unsigned long long* part_stats;  // kWordInserts / kWordArrivals slots
    unsigned int* faults;
};

enum : unsigned int { kFaultNext = 4u };  // an agent's position left the bucket its count used

// Per-workgroup counts of next segments.  A workgroup works on segment
// g_local of a table of n_local segments (global index seg_first + g_local);
// its agents' next buckets lie within the window margin of that segment, so
// nh[d + kNextReach] counts those d segments away (cyclically) and farther
// ones go straight to the global counts.  next_flush adds nh to them.
constexpr int kNextReach = 2;
struct NextCount {
    uint32_t* nh;  // LDS [2 kNextReach + 1]
    SegCounts next;
    uint32_t g_local, n_local, seg_first, seg_log;
};

// Wave-level (every lane of the wave calls it; inactive ones with
// active = false): counts the next buckets of the active lanes.
__device__ __forceinline__ void next_add(const NextCount& nc, uint32_t bucket, bool active) {
    const uint32_t ls = bucket >> nc.seg_log;
    const bool own = active && ls == nc.g_local;
    const unsigned long long om = __ballot(own);
    if (own && static_cast<int>(__lane_id()) == __ffsll(static_cast<long long>(om)) - 1) {
        atomicAdd(&nc.nh[kNextReach], static_cast<uint32_t>(__popcll(om)));
    }
    int d = static_cast<int>(ls) - static_cast<int>(nc.g_local);
    const int nl = static_cast<int>(nc.n_local);
    if (2 * d > nl) d -= nl;
    if (2 * d < -nl) d += nl;
    const bool near = d >= -kNextReach && d <= kNextReach;
    // Two separate atomics of different scopes: merged into one on a selected
    // pointer they would become a flat atomic, whose completion the
    // compiler can only await with every outstanding load.
    if (active && !own && near) {
        __hip_atomic_fetch_add(&nc.nh[d + kNextReach], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    if (active && !own && !near) {
        nc.next.add(nc.seg_first + ls, 1u);
    }
}

// Workgroup-level, after a barrier: nh into the global counts.  Its first wave
// does it, and the workgroup waits for that wave: no remainders (12 of them
// took 1% of the batched move), and the counts of one group, where all are of
// one, are summed across the lanes.
__device__ __forceinline__ void next_flush(const NextCount& nc) {
    if (threadIdx.x >= 64u) {
        return;
    }
    constexpr int kCounts = 2 * kNextReach + 1;
    const int k = static_cast<int>(threadIdx.x), nl = static_cast<int>(nc.n_local);
    int l = static_cast<int>(nc.g_local) + min(k, kCounts - 1) - kNextReach;
    while (l < 0) l += nl;
    while (l >= nl) l -= nl;
    const uint32_t g = nc.seg_first + static_cast<uint32_t>(l), gg = g >> nc.next.log;
    const uint32_t v = k < kCounts ? nc.nh[k] : 0u;
    if (v) nc.next.add_seg(g, v);
    if (__ballot(gg != static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(gg)))) == 0ull) {
        uint32_t sum = v;
#pragma unroll
        for (int o = 4; o > 0; o >>= 1) sum += static_cast<uint32_t>(__shfl_xor(static_cast<int>(sum), o, 64));
        if (k == 0 && sum) nc.next.add_group(gg, sum);
    } else if (v) {
        nc.next.add_group(gg, v);
    }
}
static_assert(2 * kNextReach + 1 <= 8, "summed over eight lanes");

// The agents that may land in a segment, numbered from 0: old slots [a0, a1),
// then (LISTS) the entries of the lower neighbour's list of agents going up
// and of the upper neighbour's list of agents going down, or (windows) old
// slots [c0, c1).
constexpr uint32_t kListCap = 1024;  // list entries whose slots are kept in LDS (later ones are read again)
template <bool LISTS>
struct Window {
    uint32_t a0, a1, c0, c1;
    const uint2 *up, *down;  // first entry of the one list, last entry of the other
    uint32_t n_up, n_list;
    uint32_t* lslot;  // LDS [kListCap]
    __device__ uint32_t own() const { return a1 - a0; }
    __device__ uint32_t size() const { return own() + (LISTS ? n_list : c1 - c0); }
    __device__ uint2 entry(uint32_t e) const { return e < n_up ? up[e] : *(down - (e - n_up)); }
    // Next bucket of agent r < size(); keep: note a list entry's slot.
    __device__ uint32_t bucket(const uint32_t* __restrict__ nxt, uint32_t r, bool keep) const {
        if (!LISTS) return nxt[slot(r)];
        if (r < own()) return nxt[a0 + r];
        const uint32_t k = r - own();
        const uint2 e = entry(k);
        if (keep && k < kListCap) lslot[k] = e.x;
        return e.y;
    }
    __device__ uint32_t slot(uint32_t r) const {
        if (r < own()) return a0 + r;
        const uint32_t k = r - own();
        if (!LISTS) return c0 + k;
        return k < kListCap ? lslot[k] : entry(k).x;
    }
};

// Count pass over a window: agents whose next bucket lies in [s0, s0 + S)
// bump their LDS counter.
template <uint32_t U, uint32_t T, bool LISTS>
__device__ __forceinline__ void sorted_count(const Window<LISTS>& win, const uint32_t* __restrict__ nxt, uint32_t s0,
                                             uint32_t S, uint32_t* hist) {
    const uint32_t size = win.size();
    for (uint32_t base = 0; base < size; base += U * T) {
        uint32_t b[U];
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {
            const uint32_t r = base + u * T + threadIdx.x;
            b[u] = win.bucket(nxt, min(r, size - 1u), r < size);
        }
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {
            const uint32_t off = b[u] - s0;
            (void)wave_rank_add(hist, off, base + u * T + threadIdx.x < size && off < S);
        }
    }
}

// Lists agents that will leave the segment (LISTS).  g, above, below: the
// segment and its neighbours in its table; n: LDS [2], the two lists'
// lengths; [base, end): the segment's new slots.
struct Leavers {
    uint32_t* n;
    uint2* leave;
    uint32_t base, end;
    uint32_t g, above, below, seg_log;
    unsigned int* faults;
};

// Wave-level (every lane of the wave calls it): lists the agents of new slots
// q[u] and next buckets b[u] where active[u]; one LDS atomic per wave and
// direction.
template <uint32_t U>
__device__ __forceinline__ void leave_round(const Leavers& lv, const uint32_t (&q)[U], const uint32_t (&b)[U],
                                            const bool (&active)[U]) {
    const unsigned long long lt = (1ull << __lane_id()) - 1ull;
    unsigned long long mu[U], md[U];
    uint32_t nu = 0, nd = 0;
    bool far = false;
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
        const uint32_t s = b[u] >> lv.seg_log;
        const bool out = active[u] && s != lv.g;
        mu[u] = __ballot(out && s == lv.above);
        md[u] = __ballot(out && s != lv.above && s == lv.below);
        far = far || (out && s != lv.above && s != lv.below);
        nu += static_cast<uint32_t>(__popcll(mu[u]));
        nd += static_cast<uint32_t>(__popcll(md[u]));
    }
    if (far) {
        atomicOr(lv.faults, kFaultBinCount);  // beyond the margin: the next move would not find it
    }
    if (nu + nd == 0u) {  // wave-uniform
        return;
    }
    uint32_t au = 0, ad = 0;
    if (__lane_id() == 0) {
        au = atomicAdd(&lv.n[0], nu);
        ad = atomicAdd(&lv.n[1], nd);
    }
    au = lv.base + static_cast<uint32_t>(__shfl(static_cast<int>(au), 0, 64));
    ad = lv.end - 1u - static_cast<uint32_t>(__shfl(static_cast<int>(ad), 0, 64));
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
        if ((mu[u] >> __lane_id()) & 1ull) lv.leave[au + static_cast<uint32_t>(__popcll(mu[u] & lt))] = make_uint2(q[u], b[u]);
        if ((md[u] >> __lane_id()) & 1ull) lv.leave[ad - static_cast<uint32_t>(__popcll(md[u] & lt))] = make_uint2(q[u], b[u]);
        au += static_cast<uint32_t>(__popcll(mu[u]));
        ad -= static_cast<uint32_t>(__popcll(md[u]));
    }
}

// Workgroup-level, after a barrier: adds the next segments of `placed` agents
// to the next move's counts, of whom the lists received lv.n less n0 (up)
// and n1 (down); the rest stay.
__device__ __forceinline__ void leave_flush(const Leavers& lv, const SegCounts& next, uint32_t seg_first,
                                            uint32_t placed, uint32_t n0, uint32_t n1) {
    const uint32_t up = lv.n[0] - n0, down = lv.n[1] - n1, stay = placed - up - down;
    const uint32_t own = (seg_first + lv.g) >> next.log, above = (seg_first + lv.above) >> next.log,
                   below = (seg_first + lv.below) >> next.log;
    if (threadIdx.x == 0u) {  // its group's sum takes the neighbours of the same group along
        const uint32_t sum = stay + (above == own ? up : 0u) + (below == own ? down : 0u);
        if (stay) next.add_seg(seg_first + lv.g, stay);
        if (sum) next.add_group(own, sum);
    }
    if (threadIdx.x == 1u && up) {
        next.add_seg(seg_first + lv.above, up);
        if (above != own) next.add_group(above, up);
    }
    if (threadIdx.x == 2u && down) {
        next.add_seg(seg_first + lv.below, down);
        if (below != own) next.add_group(below, down);
    }
}

__device__ __forceinline__ Leavers leavers_of(const SortedMove& mv, const NextCount& nc, uint32_t base, uint32_t end) {
    return Leavers{nc.nh, mv.to.leave, base, end, nc.g_local, nc.g_local + 1u == nc.n_local ? 0u : nc.g_local + 1u,
                   nc.g_local ? nc.g_local - 1u : nc.n_local - 1u, nc.seg_log, mv.faults};
}

// Hot state of the agent in one old slot: next bucket, position, target,
// speed and caller index.
struct HotAgent {
    float2 p, tg;
    float sp;
    uint32_t h, b;
};

// The agent of old slot k, whose next bucket (counted for its placement) is
// `bucket`.
template <bool UNIFORM>
__device__ __forceinline__ HotAgent load_agent(const SortedMove& mv, uint32_t k, uint32_t bucket) {
    const SortedBufs& src = mv.src;
    HotAgent a;
    a.b = bucket;
    a.p = src.pos[k];
    const uint4 r = src.rec[k];
    a.tg = make_float2(__uint_as_float(r.x), __uint_as_float(r.y));
    a.sp = UNIFORM ? mv.spd_const : __uint_as_float(r.z);
    a.h = r.w;
    return a;
}

// Steps an agent (random_move.comp:841-852) and stores it at new slot q; for
// an arrival, what the route choice decides (target, next bucket, heading)
// is left to k_route_sorted, and rec / rec_spd receive its arrival record.
// Returns whether the agent arrived; n_ins counts a cell change.
template <bool UNIFORM, bool WRITE_DIR>
__device__ __forceinline__ bool step_agent(const SortedMove& mv, const TableView& t, const HotAgent& a, uint32_t q,
                                           uint32_t& n_ins, uint4& rec, float& rec_spd, uint32_t& next_bucket) {
    const SortedBufs& dst = mv.dst;
    const uint32_t b = a.b;
    const float2 p = a.p;
    const float2 tg = a.tg;
    const float sp = a.sp;
    const uint32_t h = a.h;
    const float dx = tg.x - p.x;
    const float dy = tg.y - p.y;
    const float len = vlen(dx, dy);
    float2 np = tg, d = make_float2(0.0f, 0.0f);
    const bool arr = !(len > sp);
    if (!arr) {
        const float4 w = walk_step(p.x, p.y, dx, dy, len, sp);
        np = make_float2(w.x, w.y);
        d = make_float2(w.z, w.w);
    }
    const int32_t cx = cell_coord(np.x, t.inv_cell), cy = cell_coord(np.y, t.inv_cell);
    if (bucket_of(cx, cy, t.lw, t.wmask, t.hmask) != b) {
        atomicOr(mv.faults, kFaultNext);
    }
    n_ins += (cx != cell_coord(p.x, t.inv_cell) || cy != cell_coord(p.y, t.inv_cell)) ? 1u : 0u;
    dst.pos[q] = np;
    dst.rec[q] = hot_record(tg, sp, h);  // an arrival's target is replaced by k_route_sorted
    if (!arr) {
        next_bucket = bucket_of_pos(next_position(np, tg, sp), t);
        dst.nxt[q] = next_bucket;
        if (WRITE_DIR) dst.dir[q] = d;
    }
    rec = make_uint4(q, h, __float_as_uint(np.x), __float_as_uint(np.y));
    rec_spd = sp;
    return arr;
}

// Moves the agent of old slot k, counted in `bucket`, to new slot q
// (load_agent, then step_agent).
template <bool UNIFORM, bool WRITE_DIR>
__device__ __forceinline__ bool move_agent(const SortedMove& mv, const TableView& t, uint32_t k, uint32_t bucket,
                                           uint32_t q, uint32_t& n_ins, uint4& rec, float& rec_spd,
                                           uint32_t& next_bucket) {
    return step_agent<UNIFORM, WRITE_DIR>(mv, t, load_agent<UNIFORM>(mv, k, bucket), q, n_ins, rec, rec_spd,
                                          next_bucket);
}

// Appends one arrival record at list index i.
template <bool UNIFORM>
__device__ __forceinline__ void put_arrival(const SortedMove& mv, uint32_t i, const uint4& rec, float spd) {
    mv.arr_rec[i] = rec;
    if (!UNIFORM) mv.arr_spd[i] = spd;
}

// Wave-level: the next segment of one placed agent per lane.
template <bool LISTS>
__device__ __forceinline__ void next_one(const NextCount& nc, const Leavers& lv, uint32_t q, uint32_t bucket,
                                         bool active) {
    if (LISTS) {
        const uint32_t qs[1] = {q}, bs[1] = {bucket};
        const bool as[1] = {active};
        leave_round<1>(lv, qs, bs, as);
    } else {
        next_add(nc, bucket, active);
    }
}

// Rank pass over a window: each agent whose next bucket lies in the segment
// takes cursor[bucket]++, its new slot.  The segment's output position j = slot - base records the
// agent's window index in map[j] and its bucket in the segment in mapb[j]
// when j < cap; past cap (a segment more
// crowded than the map holds) the agent is moved and stored at once.  A
// position at or past limit (the slots the segment was given) is a count
// mismatch: the agent is not stored and kFaultBinCount is raised.  Reads
// only the next buckets; the next round's are loaded before this round is
// ranked.  Waves run the rounds independently (the rank helper needs whole
// waves, no workgroup barrier).
template <uint32_t U, uint32_t T, bool UNIFORM, bool WRITE_DIR, bool LISTS>
__device__ __forceinline__ void sorted_rank(const SortedMove& mv, const TableView& t, const NextCount& nc,
                                            const Leavers& lv, const Window<LISTS>& win, uint32_t s0,
                                            uint32_t* cursor, uint16_t* map, uint16_t* mapb, uint32_t base,
                                            uint32_t cap, uint32_t limit, uint32_t* arr_count, uint32_t arr_base,
                                            uint32_t& n_ins) {
    const uint32_t size = win.size();
    if (size == 0u) {
        return;
    }
    const uint32_t S = 1u << t.seg_log;
    uint32_t bn[U];
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
        bn[u] = win.bucket(mv.src.nxt, min(u * T + threadIdx.x, size - 1u), false);
    }
    for (uint32_t r0 = 0; r0 < size; r0 += U * T) {
        uint32_t b[U];
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {
            b[u] = bn[u];
        }
        if (r0 + U * T < size) {
#pragma unroll
            for (uint32_t u = 0; u < U; u++) {
                bn[u] = win.bucket(mv.src.nxt, min(r0 + U * T + u * T + threadIdx.x, size - 1u), false);
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {
            const uint32_t k = r0 + u * T + threadIdx.x;
            const bool mine = k < size && b[u] - s0 < S;
            const uint32_t j = wave_rank_add(cursor, b[u] - s0, mine) - base;
            bool moved = false, arr = false;
            uint32_t nb = 0;
            if (mine) {
                uint4 rec;
                float rs;
                if (j >= limit) {
                    atomicOr(mv.faults, kFaultBinCount);
                } else if (j < cap) {
                    map[j] = static_cast<uint16_t>(k);
                    mapb[j] = static_cast<uint16_t>(b[u] - s0);
                } else {
                    moved = true;
                    arr = move_agent<UNIFORM, WRITE_DIR>(mv, t, win.slot(k), b[u], base + j, n_ins, rec, rs, nb);
                    if (arr) put_arrival<UNIFORM>(mv, arr_base + atomicAdd(arr_count, 1u), rec, rs);
                }
            }
            next_one<LISTS>(nc, lv, base + j, nb, moved && !arr);
        }
    }
}

// Store pass over the segment's first min(total, cap) new slots, in slot
// order: each agent's state is gathered from its old slot (the window index
// in map; its bucket, s0 + mapb, needs no gather), moved and stored, so every wave writes consecutive slots and each
// output line is written whole.  A round's U gathers are all issued before
// the first agent is stepped (its stores would otherwise hold back the
// next agent's loads).  Arrivals are listed for k_route_sorted (one LDS
// atomic per wave and round).
template <uint32_t U, uint32_t T, bool UNIFORM, bool WRITE_DIR, bool LISTS>
__device__ __forceinline__ void sorted_store(const SortedMove& mv, const TableView& t, const NextCount& nc,
                                             const Leavers& lv, const Window<LISTS>& win, const uint16_t* map,
                                             const uint16_t* mapb,
                                             uint32_t s0, uint32_t base, uint32_t count,
                                             uint32_t* arr_count, uint32_t arr_base, uint32_t& n_ins) {
    const unsigned long long lt = (1ull << __lane_id()) - 1ull;
    for (uint32_t j0 = 0; j0 < count; j0 += U * T) {
        bool arr[U];
        uint4 rec[U];
        float rs[U];
        HotAgent ag[U];
        uint32_t nb[U], q[U];
        bool stays[U];
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {  // j0 < count: slot count - 1 is mapped
            const uint32_t j = min(j0 + u * T + threadIdx.x, count - 1u);
            ag[u] = load_agent<UNIFORM>(mv, win.slot(map[j]), s0 + mapb[j]);
        }
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {
            const uint32_t j = j0 + u * T + threadIdx.x;
            arr[u] = false;
            nb[u] = 0;
            q[u] = base + j;
            if (j < count) {
                arr[u] = step_agent<UNIFORM, WRITE_DIR>(mv, t, ag[u], q[u], n_ins, rec[u], rs[u], nb[u]);
            }
            stays[u] = j < count && !arr[u];
            if (!LISTS) next_add(nc, nb[u], stays[u]);
        }
        if (LISTS) leave_round<U>(lv, q, nb, stays);
        unsigned long long am[U];
        uint32_t round_arr = 0;
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {
            am[u] = __ballot(arr[u]);
            round_arr += static_cast<uint32_t>(__popcll(am[u]));
        }
        if (round_arr) {  // wave-uniform
            uint32_t at = 0;
            if (__lane_id() == 0) at = atomicAdd(arr_count, round_arr);
            at = arr_base + static_cast<uint32_t>(__shfl(static_cast<int>(at), 0, 64));
#pragma unroll
            for (uint32_t u = 0; u < U; u++) {
                if (arr[u]) {
                    put_arrival<UNIFORM>(mv, at + static_cast<uint32_t>(__popcll(am[u] & lt)), rec[u], rs[u]);
                }
                at += static_cast<uint32_t>(__popcll(am[u]));
            }
        }
    }
}

// Order of the segments' workgroups: three move workgroups of 512 threads and
// 50 KB of LDS share a CU.  The route choice takes the same order, so that a
// segment's arrival records are in the L2 of the XCD that reads them.
__device__ __forceinline__ uint32_t seg_order(uint32_t bid, uint32_t n_seg) {
    return xcd_deal<4>(bid, n_seg, 3u * kCus);
}

// Move workgroups have 512 threads; where each gets a CU of its own, 1,024
// with one slot per thread and round: the phases of a lone workgroup are a
// chain of waits, and twice the threads take half the rounds.  Ticks, us: 100k
// agents on 64 segments of 2^11 buckets 22.7 -> 19.5; 1M on 256 of 2^12 43.6 ->
// 39.2; but 1M on 512 of 2^11, two workgroups a CU, 37.8 -> 41.9.
constexpr uint32_t kSortedThreads = 512, kSortedWide = 1024;
inline bool one_move_per_cu(uint32_t n_seg, uint32_t smallest_seg_log) {
    return n_seg <= kCus && (1u << smallest_seg_log) >= kSortedWide;  // a thread scans at least one bucket
}

// Waves a SIMD has to have room for: two workgroups a CU with eight slots per
// thread (the lists' two more registers, 130, had left one: 1M agents on 512
// segments 58 -> 64 us).
constexpr uint32_t sorted_waves(uint32_t unroll) { return unroll == 8u ? 4u : 1u; }

// LDS of the sorted move: the segment's counters (4 bytes per bucket) and,
// for its first sorted_map_cap new slots, each agent's window index and its
// bucket in the segment (2 + 2 bytes).  Segments of up to 2^12 buckets map 2
// slots per bucket (12 bytes per bucket in all), larger ones 1 (8 bytes).
// The slots of list entries follow the maps.
__host__ __device__ constexpr uint32_t sorted_map_cap(uint32_t seg_log) {
    return seg_log <= 12u ? (2u << seg_log) : (1u << seg_log);
}
__host__ __device__ constexpr size_t sorted_lds_bytes(uint32_t seg_log) {
    return (size_t{4} << seg_log) + size_t{4} * sorted_map_cap(seg_log) + size_t{4} * kListCap;
}

// Count and place segment g (global index; s0 its first bucket in table t).
// Writes the segment's absolute bucket offsets to start_out[s0 + j];
// *base_out / *total_out receive the segment's first slot and agent count
// (all threads).  The segment's insert and arrival counts go to the
// statistics slots; its agents' next segments are counted for the next move.
template <uint32_t U, uint32_t T, bool UNIFORM, bool WRITE_DIR, bool LISTS>
__device__ __forceinline__ void sorted_segment(const SortedMove& mv, const TableView& t, const NextCount& nc,
                                               uint32_t s0, uint32_t g, uint32_t* hist, uint32_t* lds,
                                               uint32_t* sh, uint32_t* __restrict__ start_out, uint32_t* base_out,
                                               uint32_t* total_out) {
    const uint32_t tid = threadIdx.x;
    const uint32_t S = 1u << t.seg_log;
    // the counts before the segment, or its scanned slots: loaded while the window is counted
    uint32_t before = 0, st0 = 0, st1 = 0;
    if (mv.cur.seg) {
        before = mv.cur.before(g, tid, T);
        st1 = mv.cur.seg[g];
    } else {
        st0 = mv.seg_start[g];
        st1 = mv.seg_start[g + 1];
    }
    for (uint32_t j = tid; j < S; j += T) {
        hist[j] = 0u;
    }
    if (tid < 2 * kNextReach + 1) {
        nc.nh[tid] = 0u;
    }
    if (tid == 0) {
        sh[0] = 0u;  // the segment's arrivals so far
    }
    __syncthreads();
    uint16_t* map = reinterpret_cast<uint16_t*>(hist + S);
    uint16_t* mapb = map + sorted_map_cap(t.seg_log);
    Window<LISTS> win{};
    if (LISTS) {
        const uint32_t first = g - nc.g_local;
        const Leavers at = leavers_of(mv, nc, 0u, 0u);
        const uint4 me = mv.from.rec[g], lo = mv.from.rec[first + at.below], hi = mv.from.rec[first + at.above];
        win.a0 = me.x;
        win.a1 = me.y;
        win.up = mv.from.leave + lo.x;
        win.down = mv.from.leave + hi.y - 1;
        win.n_up = nc.n_local > 1u ? lo.z : 0u;
        win.n_list = win.n_up + (nc.n_local > 1u ? hi.w : 0u);
        win.lslot = reinterpret_cast<uint32_t*>(mapb + sorted_map_cap(t.seg_log));
    } else {
        bin_window(t, s0, win.a0, win.a1, win.c0, win.c1);
    }
    const uint32_t wsize = win.size();
    // A window of at most R T slots is counted in one round whose LDS
    // atomics also give each agent its rank in its bucket (kept in
    // registers, so no rank pass is needed); larger windows are counted,
    // then ranked, in rounds.
    // (U <= 4: 3 U slots per thread, 6,144 per round at U = 4, so that more
    // windows take one round; the registers stay within the same occupancy)
    constexpr uint32_t R = U <= 4 ? 3 * U : 2 * U;
    const bool one_round = wsize <= R * T;  // workgroup-uniform
    // (bucket offset << 16) | rank in the bucket, ~0 when not the segment's
    // agent (segments have at most 2^14 buckets, windows here R T <= 2^13 slots)
    uint32_t pk[R];
    if (one_round) {
        uint32_t b[R];
#pragma unroll
        for (uint32_t r = 0; r < R; r++) {
            const uint32_t idx = r * T + tid;
            b[r] = idx < wsize ? win.bucket(mv.src.nxt, idx, true) : 0u;
        }
#pragma unroll
        for (uint32_t r = 0; r < R; r++) {
            const uint32_t off = b[r] - s0;
            const bool mine = r * T + tid < wsize && off < S;
            const uint32_t rank = wave_rank_add(hist, off, mine);
            pk[r] = mine ? (off << 16) | rank : ~0u;
        }
    } else {
        sorted_count<2 * U, T>(win, mv.src.nxt, s0, S, hist);
    }
    if (mv.cur.seg) {
        before = wave_sum(before);
        if (__lane_id() == 0) sh[1 + (tid >> 6)] = before;
    }
    __syncthreads();
    if (mv.cur.seg) {
        for (uint32_t w = 0; w < T / 64; w++) st0 += sh[1 + w];
        st1 += st0;
    }
    const uint32_t per = S / T;
    uint32_t run = 0;
    for (uint32_t q = 0; q < per; q++) {
        run += hist[tid * per + q];
    }
    uint32_t total = 0;
    uint32_t excl = block_excl_scan<T>(run, lds, total);
    // the slots this segment was given, clamped to [0, n): counts that went
    // wrong raise a fault but never place an agent outside the state
    const uint32_t base = min(st0, mv.n);
    const uint32_t end = max(base, min(st1, mv.n));
    const uint32_t limit = end - base;
    if (tid == 0 && total != limit) {
        atomicOr(mv.faults, kFaultBinCount);
    }
    if (tid == 0 && mv.cur.seg) mv.seg_start[g] = base;
    for (uint32_t q = 0; q < per; q++) {  // counts -> absolute bucket offsets
        const uint32_t v = hist[tid * per + q];
        hist[tid * per + q] = base + excl;
        excl += v;
    }
    __syncthreads();
    // the offsets into the new bucket table, clamped to the segment's slots,
    // stored in bucket order (whole lines per wave)
    for (uint32_t j = tid; j < S; j += T) {
        start_out[s0 + j] = min(hist[j], base + limit);
    }
    uint32_t n_ins = 0;
    const Leavers lv = leavers_of(mv, nc, base, end);
    // window indices must fit the map's 16 bits; a window past that moves
    // every agent straight from the rank pass
    const uint32_t cap = wsize <= 65536u ? sorted_map_cap(t.seg_log) : 0u;
    if (one_round) {
#pragma unroll
        for (uint32_t r = 0; r < R; r++) {
            const uint32_t idx = r * T + tid;
            bool moved = false, arr = false;
            uint32_t nb = 0, q = 0;
            if (pk[r] != ~0u) {
                const uint32_t j = hist[pk[r] >> 16] - base + (pk[r] & 0xffffu);
                q = base + j;
                if (j >= limit) {
                    atomicOr(mv.faults, kFaultBinCount);
                } else if (j < cap) {
                    map[j] = static_cast<uint16_t>(idx);
                    mapb[j] = static_cast<uint16_t>(pk[r] >> 16);
                } else {
                    uint4 rec;
                    float rs;
                    moved = true;
                    arr = move_agent<UNIFORM, WRITE_DIR>(mv, t, win.slot(idx), s0 + (pk[r] >> 16), base + j, n_ins,
                                                         rec, rs, nb);
                    if (arr) put_arrival<UNIFORM>(mv, base + atomicAdd(&sh[0], 1u), rec, rs);
                }
            }
            next_one<LISTS>(nc, lv, q, nb, moved && !arr);
        }
    } else {
        __syncthreads();  // the rank pass advances the offsets the stores above read
        sorted_rank<U, T, UNIFORM, WRITE_DIR, LISTS>(mv, t, nc, lv, win, s0, hist, map, mapb, base, cap, limit,
                                                     &sh[0], base, n_ins);
    }
    __syncthreads();
    sorted_store<U, T, UNIFORM, WRITE_DIR, LISTS>(mv, t, nc, lv, win, map, mapb, s0, base,
                                                  min(min(total, cap), limit), &sh[0], base, n_ins);
    __syncthreads();
    if (LISTS) {
        leave_flush(lv, nc.next, g - nc.g_local, min(total, limit) - sh[0], 0u, 0u);
        if (tid == 0) mv.to.rec[g] = make_uint4(base, end, lv.n[0], lv.n[1]);
    } else {
        next_flush(nc);
    }
    // block totals of insertions and arrivals, one slot update each
    const uint32_t si = block_sum<T>(n_ins, lds);
    if (tid == 0) {
        const uint32_t sa = sh[0];
        slot_add(mv.part_stats, g, kWordInserts, si);
        slot_add(mv.part_stats, g, kWordArrivals, sa);
        mv.seg_arr[g] = sa;
    }
    *base_out = base;
    *total_out = limit;
}


// Sorted move of one table (grid: n_seg workgroups, after kXcds more when the
// previous tick's statistics are pending; dynamic LDS:
// sorted_lds_bytes(seg_log)).
template <uint32_t U, uint32_t T, bool UNIFORM, bool WRITE_DIR, bool LISTS>
static __global__ __launch_bounds__(T, sorted_waves(U)) void k_move_sorted(SortedMove mv, BinDev b, TickFinish fin) {
    extern __shared__ uint32_t hist[];
    __shared__ uint32_t lds[T / 64];
    __shared__ uint32_t nh[2 * kNextReach + 1];
    __shared__ uint32_t sh[1 + T / 64];
    const uint32_t extra = gridDim.x - b.n_seg;
    if (blockIdx.x < extra) {  // the previous tick's statistics, beside the move
        fin.run(blockIdx.x);
        return;
    }
    const uint32_t seg = seg_order(blockIdx.x - extra, b.n_seg);
    const NextCount nc{nh, mv.next, seg, b.n_seg, 0u, b.seg_log};
    uint32_t base, total;
    sorted_segment<U, T, UNIFORM, WRITE_DIR, LISTS>(mv, table_view(b), nc, seg << b.seg_log, seg, hist, lds, sh,
                                             b.new_start, &base, &total);
    if (seg == b.n_seg - 1 && threadIdx.x == 0) {
        b.new_start[b.m] = base + total;
        if (base + total != b.n) {
            atomicOr(mv.faults, kFaultBinCount);
        }
    }
}

// First slot of every segment from the per-segment agent counts (the
// segments of all tables in order): seg_start[g] = cnt[0] + ... + cnt[g - 1],
// seg_start[n_seg] = the total, which must be n.  cnt and its group sums are
// cleared for their next use.  One workgroup: wave w takes the contiguous chunk [w C, (w + 1) C) in
// pieces of 64 K entries, each loaded at once (coalesced, K loads in flight
// per lane) and kept in registers for both the chunk sum and the offsets.
template <uint32_t T>
static __global__ __launch_bounds__(T) void k_seg_scan(uint32_t* __restrict__ cnt, uint32_t* __restrict__ group,
                                                       uint32_t group_words, uint32_t* __restrict__ seg_start,
                                                       uint32_t n_seg, uint32_t n, unsigned int* faults) {
    constexpr uint32_t W = T / 64, K = 16;
    __shared__ uint32_t wsum[W];
    const uint32_t lane = __lane_id(), w = threadIdx.x >> 6;
    const uint32_t C = (n_seg + W - 1) / W;
    const uint32_t c0 = min(w * C, n_seg), c1 = min(c0 + C, n_seg);
    const bool one_piece = C <= 64u * K;  // workgroup-uniform
    uint32_t v[K];
    uint32_t part = 0;
    for (uint32_t p0 = c0; p0 < c1; p0 += 64u * K) {
#pragma unroll
        for (uint32_t k = 0; k < K; k++) {
            const uint32_t g = p0 + 64u * k + lane;
            v[k] = g < c1 ? cnt[g] : 0u;
        }
#pragma unroll
        for (uint32_t k = 0; k < K; k++) {
            part += v[k];
        }
    }
    part = wave_sum(part);
    if (lane == 0) wsum[w] = part;
    __syncthreads();
    uint32_t run = 0, total = 0;
    for (uint32_t k = 0; k < W; k++) {
        run += (k < w) ? wsum[k] : 0u;
        total += wsum[k];
    }
    for (uint32_t p0 = c0; p0 < c1; p0 += 64u * K) {
        if (!one_piece) {
#pragma unroll
            for (uint32_t k = 0; k < K; k++) {
                const uint32_t g = p0 + 64u * k + lane;
                v[k] = g < c1 ? cnt[g] : 0u;
            }
        }
#pragma unroll
        for (uint32_t k = 0; k < K; k++) {
            const uint32_t g = p0 + 64u * k + lane;
            const uint32_t inc = wave_incl_scan(v[k]);
            if (g < c1) {
                seg_start[g] = run + inc - v[k];
                cnt[g] = 0u;
            }
            run += static_cast<uint32_t>(__shfl(static_cast<int>(inc), 63, 64));
        }
    }
    for (uint32_t k = threadIdx.x; k < group_words; k += T) {
        group[k] = 0u;
    }
    if (threadIdx.x == 0) {
        seg_start[n_seg] = total;
        if (total != n) {
            atomicOr(faults, kFaultBinCount);
        }
    }
}

// Route choice of the arrivals listed by the sorted move: one workgroup per
// segment (grid n_seg), its list at arr_rec[seg_start[g] ...].  An arrival
// stands on its old target (the position in its record); the route choice
// (random_move.comp:778-828) updates the caller-order route state and gives
// the new target, the bucket of the next move and (last tick of a batch) the
// heading.
template <bool UNIFORM, bool WRITE_DIR, bool LISTS>
__device__ __forceinline__ void route_segment_list(const SortedMove& mv, const TableView& t, const NextCount& nc,
                                                   uint32_t g) {
    const SortedBufs& dst = mv.dst;
    const uint4 sr = LISTS ? mv.to.rec[g] : make_uint4(0u, 0u, 0u, 0u);
    const uint32_t base = LISTS ? sr.x : min(mv.seg_start[g], mv.n), cnt = mv.seg_arr[g];
    const Leavers lv = leavers_of(mv, nc, base, sr.y);
    if (threadIdx.x < 2 * kNextReach + 1) {
        nc.nh[threadIdx.x] = !LISTS || threadIdx.x > 1u ? 0u : (threadIdx.x ? sr.w : sr.z);
    }
    __syncthreads();
    for (uint32_t j0 = 0; j0 < cnt; j0 += blockDim.x) {  // whole-block rounds: next_add is wave-level
        const uint32_t j = j0 + threadIdx.x;
        uint32_t nb = 0, q = 0;
        if (j < cnt) {
            const uint4 a = mv.arr_rec[base + j];
            const uint32_t hh = a.y;
            q = a.x;
            const float2 at = make_float2(__uint_as_float(a.z), __uint_as_float(a.w));
            const float s = UNIFORM ? mv.spd_const : mv.arr_spd[base + j];
            const uint4 w = mv.cold[2u * hh];
            uint4 st = mv.cold[2u * hh + 1u];
            float2 nt = at;
            uint32_t r = w.x;
            uint2 c = make_uint2(w.y, w.z);
            choose_route_at(nt, r, c, st, mv.roads, mv.conns);
            mv.cold[2u * hh] = cold_word(r, c);
            mv.cold[2u * hh + 1u] = st;
            nb = bucket_of_pos(next_position(at, nt, s), t);
            *reinterpret_cast<float2*>(&dst.rec[q]) = nt;  // the record's target
            dst.nxt[q] = nb;
            if (WRITE_DIR) dst.dir[q] = heading(nt, at, s);
        }
        next_one<LISTS>(nc, lv, q, nb, j < cnt);
    }
    __syncthreads();
    if (LISTS) {
        leave_flush(lv, nc.next, g - nc.g_local, cnt, sr.z, sr.w);
        if (threadIdx.x == 0) mv.to.rec[g] = make_uint4(sr.x, sr.y, lv.n[0], lv.n[1]);
    } else {
        next_flush(nc);
    }
}

template <bool UNIFORM, bool WRITE_DIR, bool LISTS>
static __global__ __launch_bounds__(kBlock) void k_route_sorted(SortedMove mv, BinDev b) {
    __shared__ uint32_t nh[2 * kNextReach + 1];
    const uint32_t g = seg_order(blockIdx.x, gridDim.x);
    route_segment_list<UNIFORM, WRITE_DIR, LISTS>(mv, table_view(b), NextCount{nh, mv.next, g, b.n_seg, 0u, b.seg_log}, g);
}

// Route choice and neighbour pass in one launch (run_ticks only).  Neither
// reads what the other writes: the neighbour pass needs the positions and
// bucket offsets the move left, the route choice rewrites targets, next
// buckets and route state.  Groups of kXcds workgroups (one per XCD) are
// dealt to the two in turn while both have some left: a route workgroup
// waits on random cache lines most of its time, and spreading the routes
// through the whole launch made it as long as their chain of waits.
// Measured (kernel trace, us; apart -> together in turn): 8M agents
// 55 + 77 -> 131 (129 with all routes first, 142 spread evenly), 64
// scenarios of 5.8M agents 33 + 77 -> 99 (103, 93 to 104), 1M agents
// 4.9 + 13.0 -> 16.4 (16.9, 17.3).
struct RouteMix {
    uint32_t n_route, n_collide;
    __host__ __device__ static uint32_t groups(uint32_t n) { return (n + kXcds - 1u) / kXcds; }
    __host__ uint32_t blocks() const { return kXcds * (groups(n_route) + groups(n_collide)); }
    // Workgroup bid's part: route workgroup r, or neighbour workgroup r (r may
    // lie past the last one).
    __device__ bool routes(uint32_t bid, uint32_t& r) const {
        const uint32_t grp = bid / kXcds, rg = groups(n_route), cg = groups(n_collide);
        const uint32_t both = 2u * min(rg, cg);
        r = (grp < both ? grp / 2u : grp - both / 2u) * kXcds + bid % kXcds;
        return grp < both ? (grp & 1u) == 0u : rg > cg;
    }
};

template <bool UNIFORM, int P, bool LISTS>
static __global__ __launch_bounds__(kBlock, 8) void k_route_collide(SortedMove mv, BinDev b, AgentsDev a, GridDev g,
                                                                    const float2* __restrict__ bpos,
                                                                    unsigned long long* __restrict__ part_pairs,
                                                                    RouteMix mix) {
    __shared__ uint32_t lds[kBlock / 64];
    __shared__ uint32_t nh[2 * kNextReach + 1];
    __shared__ float2 stage_all[kBlock / 64 * kStage];
    uint32_t r;
    if (mix.routes(blockIdx.x, r)) {
        if (r >= mix.n_route) return;
        const uint32_t seg = seg_order(r, mix.n_route);
        // the counts this tick's move consumed, cleared for the move after next
        if (threadIdx.x == 0) mv.cur.clear(seg);
        route_segment_list<UNIFORM, false, LISTS>(mv, table_view(b), NextCount{nh, mv.next, seg, b.n_seg, 0u, b.seg_log},
                                           seg);
    } else {
        if (r >= mix.n_collide) return;
        collide_block<P>(a, g, bpos, part_pairs, collide_order(r, mix.n_collide), lds, stage_all);
    }
}

// Wave-level: one count per distinct segment among the active lanes' gseg
// (the lanes of a wave hold consecutive slots in bucket order, so there are
// few).
__device__ __forceinline__ void count_next_segment(const SegCounts& next, uint32_t gseg, bool active) {
    unsigned long long todo = __ballot(active);
    while (todo) {
        const int leader = __ffsll(static_cast<long long>(todo)) - 1;
        const uint32_t k = static_cast<uint32_t>(__shfl(static_cast<int>(gseg), leader, 64));
        const unsigned long long peers = __ballot(active && gseg == k) & todo;
        if (static_cast<int>(__lane_id()) == leader) {
            next.add(k, static_cast<uint32_t>(__popcll(peers)));
        }
        todo &= ~peers;
    }
}

// Entering the sorted state (LISTS): lists the agent of slot q, in segment gl
// of n_seg, if its next bucket lies in another segment.
__device__ __forceinline__ void init_leave(const SegLists& to, unsigned int* faults, uint32_t q, uint32_t bucket,
                                           uint32_t gl, uint32_t n_seg, uint32_t seg_log) {
    const uint32_t s = bucket >> seg_log;
    if (s == gl) {
        return;
    }
    uint4* r = &to.rec[gl];
    if (s == (gl + 1u == n_seg ? 0u : gl + 1u)) {
        to.leave[r->x + atomicAdd(&r->z, 1u)] = make_uint2(q, bucket);
    } else if (s == (gl ? gl - 1u : n_seg - 1u)) {
        to.leave[r->y - 1u - atomicAdd(&r->w, 1u)] = make_uint2(q, bucket);
    } else {
        atomicOr(faults, kFaultBinCount);
    }
}

// Entering the sorted state (LISTS): the segments' slots, both lists empty.
static __global__ __launch_bounds__(kBlock) void k_seg_records(SegLists to, const uint32_t* __restrict__ start,
                                                               uint32_t n_seg, uint32_t seg_log) {
    const uint32_t g = blockIdx.x * kBlock + threadIdx.x;
    if (g < n_seg) {
        to.rec[g] = make_uint4(start[g << seg_log], start[(g + 1u) << seg_log], 0u, 0u);
    }
}

// nxt for every slot of one table: the bucket of the agent's next position;
// next (cleared before) counts them per segment, and to (LISTS; null
// otherwise, records initialised) lists those that leave theirs.
template <bool UNIFORM>
static __global__ __launch_bounds__(kBlock) void k_sorted_next(SortedBufs st, uint32_t n, float spd_const,
                                                               float inv_cell, uint32_t lw, uint32_t wmask,
                                                               uint32_t hmask, uint32_t seg_log,
                                                               SegCounts next, SegLists to, uint32_t n_seg,
                                                               unsigned int* faults) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    uint32_t b = 0;
    if (i < n) {
        const uint4 r = st.rec[i];
        const float2 p = st.pos[i];
        const float2 np = next_position(p, make_float2(__uint_as_float(r.x), __uint_as_float(r.y)),
                                        UNIFORM ? spd_const : __uint_as_float(r.z));
        b = bucket_of(cell_coord(np.x, inv_cell), cell_coord(np.y, inv_cell), lw, wmask, hmask);
        st.nxt[i] = b;
        if (to.rec) {
            const uint32_t at = bucket_of(cell_coord(p.x, inv_cell), cell_coord(p.y, inv_cell), lw, wmask, hmask);
            init_leave(to, faults, i, b, at >> seg_log, n_seg, seg_log);
        }
    }
    count_next_segment(next, b >> seg_log, i < n);
}

// p[0, n) = v (in graphs too, where memset nodes are avoided).
static __global__ __launch_bounds__(kBlock) void k_fill_u32(uint32_t* __restrict__ p, uint32_t v, uint32_t n) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) {
        p[i] = v;
    }
}

// Route state into caller order: cold[perm[i]] from slot i's road, PRNG
// state and target.
static __global__ __launch_bounds__(kBlock) void k_cold_enter(const uint32_t* __restrict__ perm,
                                                        const uint32_t* __restrict__ road,
                                                        const uint4* __restrict__ rng,
                                                        const float2* __restrict__ tgt,
                                                        const msim_road* __restrict__ roads, uint4* __restrict__ cold,
                                                        uint32_t n) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) {
        return;
    }
    const uint32_t h = perm[i], r = road[i];
    Endpoint s, e;
    load_road(roads, r, s, e);
    cold[2u * h] = cold_word(r, route_endpoint(s, e, tgt[i]));
    cold[2u * h + 1u] = rng[i];
}

// Route state back into slot order: road[i], rng[i] of caller perm[i].
static __global__ __launch_bounds__(kBlock) void k_cold_publish(const uint32_t* __restrict__ perm,
                                                          const uint4* __restrict__ cold,
                                                          uint32_t* __restrict__ road, uint4* __restrict__ rng,
                                                          uint32_t n) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) {
        return;
    }
    const uint32_t h = perm[i];
    road[i] = cold[2u * h].x;
    rng[i] = cold[2u * h + 1u];
}

// dst[i] = src[caller index of slot i], the caller index from the slot's record.
template <class V>
static __global__ __launch_bounds__(kBlock) void k_gather_rec(const uint4* __restrict__ rec,
                                                              const V* __restrict__ src, V* __restrict__ dst,
                                                              uint32_t n) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) {
        dst[i] = src[rec[i].w];
    }
}

// dst[caller index of slot i] = src[i], the caller index from the slot's record.
template <class V>
static __global__ __launch_bounds__(kBlock) void k_scatter_rec(const uint4* __restrict__ rec,
                                                               const V* __restrict__ src, V* __restrict__ dst,
                                                               uint32_t n) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) {
        dst[rec[i].w] = src[i];
    }
}

// Cells of the sorted state's agents in caller order (the caller index from
// each slot's record): k_export_cells for the sorted state.
static __global__ __launch_bounds__(kBlock) void k_export_cells_rec(const float2* __restrict__ pos,
                                                                    const uint4* __restrict__ rec, uint32_t n,
                                                                    float inv_cell, int2* __restrict__ out) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) {
        const float2 p = pos[i];
        out[rec[i].w] = make_int2(cell_coord(p.x, inv_cell), cell_coord(p.y, inv_cell));
    }
}

// k_export_state for the sorted state: target and caller index in the
// records, road and PRNG state in caller order already.
static __global__ __launch_bounds__(kBlock) void k_export_state_rec(AgentsDev a, const uint4* __restrict__ rec,
                                                                    const uint4* __restrict__ cold, uint32_t off,
                                                                    uint32_t n, uint32_t road_base, StateOut out) {
    const uint32_t j = blockIdx.x * kBlock + threadIdx.x;
    if (j >= n) {
        return;
    }
    const uint32_t k = off + j;
    const uint4 r = rec[k];
    const uint32_t i = r.w - off;
    out.pos[i] = a.pos[k];
    out.tgt[i] = make_float2(__uint_as_float(r.x), __uint_as_float(r.y));
    out.dir[i] = a.dir[k];
    out.ncount[i] = a.ncount[k];
    out.road[j] = cold[2u * k].x - road_base;
    out.rng[j] = cold[2u * k + 1u];
}

// Records from the classic per-slot arrays (entering the sorted state); spd
// nullptr: every agent moves at the constant speed.
static __global__ __launch_bounds__(kBlock) void k_pack_rec(const float2* __restrict__ tgt,
                                                            const float* __restrict__ spd,
                                                            const uint32_t* __restrict__ perm,
                                                            uint4* __restrict__ rec, uint32_t n) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) {
        rec[i] = hot_record(tgt[i], spd ? spd[i] : 0.0f, perm[i]);
    }
}

// The classic per-slot arrays from the records (readbacks, leaving the
// sorted state).
static __global__ __launch_bounds__(kBlock) void k_unpack_rec(const uint4* __restrict__ rec,
                                                              float2* __restrict__ tgt, float* __restrict__ spd,
                                                              uint32_t* __restrict__ perm, uint32_t n) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) {
        const uint4 r = rec[i];
        tgt[i] = make_float2(__uint_as_float(r.x), __uint_as_float(r.y));
        if (spd) spd[i] = __uint_as_float(r.z);
        perm[i] = r.w;
    }
}

}  // namespace msim
