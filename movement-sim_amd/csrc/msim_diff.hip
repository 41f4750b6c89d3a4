// msim_diff.hip — the differentiable tick on a batched handle and its
// hand-written adjoint.
//
// Differentiable tick (binary32, the move arithmetic of k_advance):
//   speed      s_i = v_i * theta[road_i]          (theta: per-road multiplier)
//   move       arrived: p~_i = T_i (snap; route choice as in the plain tick)
//              else:    p~_i = p_i + ((T_i - p_i) / |T_i - p_i|) * s_i
//   avoidance  p'_i = p~_i + alpha * sum_{j != i, |x_ij| < R} w(|x_ij|^2) x_ij,
//              x_ij = p~_i - p~_j, w(q) = (1 - q / R^2)^3
// over the neighbour relation of the plain collision dispatch (same exact
// predicate, same scenario tables).  theta = 1, alpha = 0 is the reference
// tick.  w, w' and w'' vanish at q = R^2, so the tick is C^2 in the positions.
//
// The adjoint freezes the discrete decisions of the forward run (arrival
// flags, targets, roads, neighbour cells): a forward pass keeps checkpoints
// (agent state and binning) every C ticks; the backward pass replays each
// segment from its checkpoint, recording per tick the pre-move positions,
// targets, roads, flags and the binning, then walks the segment backwards:
//   avoidance  lam~_k = lam_k + alpha * sum_j J(x_kj) (lam_k - lam_j),
//              J(x) = w(q) I + 2 w'(q) x x^T,   dL/dalpha += lam_k . A_k
//   move       lam_k = lam~_k - (s/L) (lam~_k - u (u . lam~_k)), u = (T-p)/L
//              dL/dtheta[road_k] += v_k (u . lam~_k);  arrived: lam_k = 0
// The reverse pass runs in binary64 on the run's binary32 values.
#include "msim_batch.hpp"

#include <cmath>
#include <cstring>

using namespace msim;

namespace msim {

// kDiffNear (on the segment tape only): the agent had a neighbour in the
// tick's avoidance.
enum DiffFlag : uint8_t { kDiffArrived = 1, kDiffNoMove = 2, kDiffNear = 4 };

struct DiffTapeDev {
    float2* pos;     // [n] position before the move
    float2* tgt;     // [n] target of the move
    uint32_t* road;  // [n] road of the move (theta index)
    uint8_t* flag;   // [n] DiffFlag bits
};

// Forward move of the differentiable tick; REPLAY takes the decisions from
// `in` instead of making them (no route choice, agent state untouched but
// for pos).  `rec` (nullable) receives the tick's decisions.
template <bool REPLAY, bool UNIFORM>
static __global__ __launch_bounds__(kBlock) void k_dadvance(AgentsDev a, const float* __restrict__ theta,
                                                     uint32_t no_move, DiffTapeDev in, DiffTapeDev rec,
                                                     const msim_road* __restrict__ roads,
                                                     const uint32_t* __restrict__ conns) {
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= a.n) {
        return;
    }
    const float2 p = a.pos[k];
    const float2 T = REPLAY ? in.tgt[k] : a.tgt[k];
    const uint32_t r = REPLAY ? in.road[k] : a.road[k];
    const float s = (UNIFORM ? a.spd_const : a.spd[k]) * theta[r];
    uint8_t flag = 0;
    float2 np = p;
    if (no_move) {
        flag = kDiffNoMove;
    } else {
        const float dx = T.x - p.x;
        const float dy = T.y - p.y;
        const float len = vlen(dx, dy);
        const bool arrived = REPLAY ? (in.flag[k] & kDiffArrived) != 0 : !(len > s);
        if (!arrived) {
            np = make_float2(p.x + (dx / len) * s, p.y + (dy / len) * s);
        } else {
            np = T;
            flag = kDiffArrived;
            if (!REPLAY) {
                float2 nt = T;
                uint32_t nr = r;
                uint4 st = a.rng[k];
                choose_route(nt, nr, st, roads, conns);
                a.tgt[k] = nt;
                a.road[k] = nr;
                a.rng[k] = st;
            }
        }
    }
    a.pos[k] = np;
    if (rec.pos) {
        rec.pos[k] = p;
        rec.tgt[k] = T;
        rec.road[k] = r;
        rec.flag[k] = flag;
    }
}

__device__ __forceinline__ float avoid_w(float q, float inv_r2) {
    const float h = 1.0f - q * inv_r2;
    return h * h * h;
}

// Arrays copied in one launch, one row of workgroups each.  Every array is a
// device allocation of its own (aligned to 16 bytes and more) of whole words.
// Small runs are bound by launches: a gradient of 3k agents over 40 ticks makes
// five such copies of 4 to 9 arrays, 2.48 ms with a transfer per array, 2.40
// with a launch per copy; at 800k agents both run at memory's rate.
constexpr uint32_t kCopyParts = 9;
constexpr uint32_t kCopyBlocks = 1024;            // workgroups per array at most
constexpr uint32_t kCopyWords = 4u * 4u * kBlock;  // words a workgroup has in flight
struct CopyParts {
    const uint32_t* src[kCopyParts];
    uint32_t* dst[kCopyParts];
    size_t words[kCopyParts];
};

static __global__ __launch_bounds__(kBlock) void k_copy_parts(CopyParts c) {
    const uint32_t part = blockIdx.y;
    const size_t words = c.words[part], quads = words / 4u;
    const uint4* __restrict__ src = reinterpret_cast<const uint4*>(c.src[part]);
    uint4* __restrict__ dst = reinterpret_cast<uint4*>(c.dst[part]);
    for (size_t q0 = static_cast<size_t>(blockIdx.x) * (kCopyWords / 4u); q0 < quads;
         q0 += static_cast<size_t>(gridDim.x) * (kCopyWords / 4u)) {
        uint4 v[4];
#pragma unroll
        for (uint32_t k = 0; k < 4u; k++) {
            const size_t q = q0 + k * kBlock + threadIdx.x;
            if (q < quads) v[k] = src[q];
        }
#pragma unroll
        for (uint32_t k = 0; k < 4u; k++) {
            const size_t q = q0 + k * kBlock + threadIdx.x;
            if (q < quads) dst[q] = v[k];
        }
    }
    const size_t tail = quads * 4u + threadIdx.x;  // the last words short of 16 bytes
    if (blockIdx.x == 0 && tail < words) {
        c.dst[part][tail] = c.src[part][tail];
    }
}

struct DiffCells {
    const BlockScen* blk;
    const ScenDev* scen;
    const uint32_t* agent_off;
    uint32_t n;
    const uint32_t* start;
    const float2* bpos;
    const uint32_t* bid;
    float inv_cell;
    float d2_limit;
    float inv_r2;
    double inv_r2_d;
    float fix_scale;   // forward avoidance: terms summed as integers in units of 1/fix_scale
    float push_allow;  // largest push per axis the rebinning windows were sized for
};

// The slots of a tick that have neighbours: each group of kNearGroup slots
// (one wave's width) lists its own, as offsets into the group.
// The adjoint of the avoidance changes nothing for the others, at the
// calibration's density four agents in five.
constexpr uint32_t kNearGroup = 64;
struct DiffNear {
    uint8_t* list;   // [n rounded up to whole groups]; nullptr: not recorded
    uint8_t* count;  // per group
    uint8_t* flag;   // [n] the tape's flags, agent order
};

// Calls f(slot) for every other slot within the d2 limit of slot s, over the
// 3x3 cells of s's scenario table.  The order of the slots inside a bucket
// follows the rebinning's LDS atomics and is not reproducible: callers sum in
// an order-independent way.
template <class F>
__device__ __forceinline__ void for_neighbours(const DiffCells& c, uint32_t s, float2 me, F&& f) {
    const BlockScen bs = c.blk[s / kBlock];
    uint32_t sid = bs.sid;
    uint32_t base = bs.start_base, lw = bs.lw, wmask = bs.wmask, hmask = bs.hmask;
    if (s >= bs.end) {
        sid++;
        while (s >= c.agent_off[sid + 1]) sid++;
        const ScenDev& sc = c.scen[sid];
        base = sc.start_base;
        lw = sc.lw;
        wmask = sc.wmask;
        hmask = sc.hmask;
    }
    const uint32_t* start = c.start + base;
    const int32_t cx = cell_coord(me.x, c.inv_cell);
    const int32_t cy = cell_coord(me.y, c.inv_cell);
    const uint32_t c0 = static_cast<uint32_t>(cx - 1) & wmask;
    const uint32_t c2 = static_cast<uint32_t>(cx + 1) & wmask;
    const bool wrap = c0 > c2;
    uint32_t lo[3], hi[3];
#pragma unroll
    for (uint32_t r = 0; r < 3u; r++) {  // the rows' bounds in one round trip
        const uint32_t rowb = (static_cast<uint32_t>(cy - 1 + static_cast<int32_t>(r)) & hmask) << lw;
        lo[r] = start[rowb + c0];
        hi[r] = start[rowb + (wrap ? wmask + 1u : c2 + 1u)];
    }
#pragma unroll
    for (uint32_t r = 0; r < 3u; r++) {
        for (uint32_t k = lo[r]; k < hi[r]; k += 2u) {  // two candidates in flight
            const float2 q0 = c.bpos[k];
            const float2 q1 = c.bpos[min(k + 1u, hi[r] - 1u)];
            if (k != s && in_range(q0, me, c.d2_limit)) f(k);
            if (k + 1u < hi[r] && k + 1u != s && in_range(q1, me, c.d2_limit)) f(k + 1u);
        }
    }
    if (wrap) {
#pragma unroll 1
        for (int32_t r = -1; r <= 1; r++) {
            const uint32_t rowb = (static_cast<uint32_t>(cy + r) & hmask) << lw;
            const uint32_t hi2 = start[rowb + c2 + 1u];
            for (uint32_t k = start[rowb]; k < hi2; k++) {
                if (k != s && in_range(c.bpos[k], me, c.d2_limit)) f(k);
            }
        }
    }
}

// Sums the pushes of a slot's neighbours; cnt counts all candidates in range
// (the slot itself among them).  A candidate whose squared distance is 0 adds
// exactly nothing (its terms are below half a unit of the sums).  The others
// wait in a short queue per slot: one lane in five has a neighbour at all, so
// summed where they are met, nearly every step of the scan would run the
// costly part for one lane or two.
template <int P>
struct PushVisitor {
    static constexpr uint32_t kQueue = 3;
    long long ix[P], iy[P];
    uint32_t cnt[P], waiting[P];
    float2 queue[P][kQueue];
    const float2 (&me)[P];
    float T, inv_r2;
    double sc;
    __device__ __forceinline__ PushVisitor(const float2 (&m)[P], const DiffCells& c)
        : me(m), T(c.d2_limit), inv_r2(c.inv_r2), sc(c.fix_scale) {
#pragma unroll
        for (int p = 0; p < P; p++) {
            ix[p] = 0;
            iy[p] = 0;
            cnt[p] = 0u;
            waiting[p] = 0u;
#pragma unroll
            for (uint32_t k = 0; k < kQueue; k++) queue[p][k] = make_float2(0.0f, 0.0f);
        }
    }
    __device__ __forceinline__ void add(int p, float2 q) {
        const float x = me[p].x - q.x;
        const float y = me[p].y - q.y;
        const float w = avoid_w(x * x + y * y, inv_r2);
        ix[p] += __double2ll_rn(static_cast<double>(w * x) * sc);
        iy[p] += __double2ll_rn(static_cast<double>(w * y) * sc);
    }
    __device__ __forceinline__ float dist2(int p, float2 q) const {  // in_range's
        const float ddx = q.x - me[p].x;
        const float ddy = q.y - me[p].y;
        return opaque(ddx * ddx) + opaque(ddy * ddy);
    }
    __device__ __forceinline__ void note(int p, float2 q, float d2) {
        cnt[p] += d2 < T ? 1u : 0u;
        if (d2 < T && d2 > 0.0f) {
            if (waiting[p] == kQueue) {
                add(p, queue[p][kQueue - 1]);
                waiting[p]--;
            }
#pragma unroll
            for (uint32_t k = kQueue - 1; k > 0; k--) queue[p][k] = queue[p][k - 1];
            queue[p][0] = q;
            waiting[p]++;
        }
    }
    __device__ __forceinline__ void one(int p, float2 q) { note(p, q, dist2(p, q)); }
    __device__ __forceinline__ void staged(int p, const float2* stage, uint32_t j0, uint32_t j1) {
        const float2* q = stage + j0;
        const float2* const pair_end = stage + (j0 + ((j1 - j0) & ~1u));
        for (; q != pair_end; q += 2) {
            const float2 q0 = q[0], q1 = q[1];
            const float d0 = dist2(p, q0), d1 = dist2(p, q1);
            note(p, q0, d0);
            note(p, q1, d1);
        }
        if ((j1 - j0) & 1u) one(p, *q);
    }
    // The sums, when all candidates were seen.
    __device__ __forceinline__ void finish() {
#pragma unroll
        for (int p = 0; p < P; p++) {
#pragma unroll
            for (uint32_t k = 0; k < kQueue; k++) {
                if (waiting[p] > k) add(p, queue[p][k]);
            }
        }
    }
};

// Forward avoidance: pos[agent] = p~ + alpha * A over the tick's binning, each
// wave staging the candidates of its 64 P slots as the neighbour pass does.
// Each binary32 term w x is rounded to a multiple of 1/fix_scale (a power of
// two with |w x| * fix_scale < 2^40, at most 2^-40 R) and the terms are
// summed as 64-bit integers, so A does not depend on the order in which the
// neighbours are visited and two runs with the same parameters are
// bit-identical.  A push beyond the windows' allowance raises kFaultBinCount
// (the run then fails instead of rebinning an agent outside its window).
// Positions without a neighbour stay as the move left them (p + 0 differs
// from p only for p = -0).
// (One slot per lane: with two, 110 registers and half the waves, 800k agents
// took 41 us against 28; a lane walking its cells in global memory, without
// staging, 33.  Seven waves a SIMD instead of six, 69 registers: a gradient of
// 800k agents over 100 ticks 15.07 -> 14.87 ms; eight spill.)
template <int P>
static __global__ __launch_bounds__(kBlock, 7) void k_davoid(DiffCells c, float alpha, float2* __restrict__ pos,
                                                             DiffNear near, unsigned int* __restrict__ faults) {
    __shared__ float2 stage_all[kBlock / 64 * kStage];
    const uint32_t blk = collide_order(blockIdx.x, gridDim.x);
    const uint32_t wave = blk * (kBlock / 64) + (threadIdx.x >> 6);
    const uint32_t w0 = wave * (64u * P);
    if (w0 >= c.n) {
        return;  // wave-uniform: no barrier follows
    }
    const uint32_t lane = __lane_id();
    const BlockScen bs = c.blk[w0 / kBlock];
    float2 me[P];
    bool valid[P];
    int32_t cx[P], cy[P];
    bool later = false;  // some valid slot lies past scenario bs.sid
#pragma unroll
    for (int p = 0; p < P; p++) {
        const uint32_t s = w0 + 64u * p + lane;
        valid[p] = s < c.n;
        me[p] = valid[p] ? c.bpos[s] : make_float2(0.0f, 0.0f);
        cx[p] = cell_coord(me[p].x, c.inv_cell);
        cy[p] = cell_coord(me[p].y, c.inv_cell);
        later = later || (valid[p] && s >= bs.end);
    }
    PushVisitor<P> v(me, c);
    if (__ballot(later) == 0ull) {
        const uint32_t last = min(64u * P, c.n - w0) - 1u;
        wave_visit_cells<P>(valid, 0u, 0u, last >> 6, last & 63u, cx, cy, c.start + bs.start_base, bs.lw, bs.wmask,
                            bs.hmask, c.bpos, stage_all + (threadIdx.x >> 6) * kStage, v);
    } else {  // across a scenario boundary: per slot
#pragma unroll
        for (int p = 0; p < P; p++) {
            const uint32_t s = w0 + 64u * p + lane;
            if (valid[p]) {
                for_neighbours(c, s, me[p], [&](uint32_t k) { v.one(p, c.bpos[k]); });
                v.cnt[p]++;  // its own
            }
        }
    }
    v.finish();
#pragma unroll
    for (int p = 0; p < P; p++) {
        const uint32_t s = w0 + 64u * p + lane;
        const bool has = valid[p] && v.cnt[p] > 1u;
        const bool moves = valid[p] && (has || me[p].x == 0.0f || me[p].y == 0.0f);
        const unsigned long long hm = __ballot(has);
        if (moves) {
            const uint32_t i = c.bid[s];
            if (near.list && has) {
                near.list[w0 + kNearGroup * p + static_cast<uint32_t>(__popcll(hm & ((1ull << lane) - 1ull)))] =
                    static_cast<uint8_t>(lane);
                near.flag[i] |= kDiffNear;
            }
            const float px = alpha * static_cast<float>(static_cast<double>(v.ix[p]) / v.sc);
            const float py = alpha * static_cast<float>(static_cast<double>(v.iy[p]) / v.sc);
            if (!(fabsf(px) <= c.push_allow) || !(fabsf(py) <= c.push_allow)) {
                atomicOr(faults, kFaultBinCount);
            }
            pos[i] = make_float2(me[p].x + px, me[p].y + py);
        }
        if (near.list && lane == 0 && w0 + kNearGroup * p < c.n) {
            near.count[wave * P + p] = static_cast<uint8_t>(__popcll(hm));
        }
    }
}

// The alpha derivative is summed into kAlphaSlots words a line apart, one
// atomic per workgroup (on one word the workgroups' atomics queue up).
constexpr uint32_t kAlphaSlots = 64, kAlphaStride = 16;

struct DiffMove {
    uint32_t n;
    const float* spd;
    float spd_const;
    const float* theta;
    DiffTapeDev tp;
    const float2* nxt_tgt;
    const uint32_t* nxt_road;
    uint32_t carry;
    double* acc;
    double* gtheta;
};

// Move adjoint of agent k, binary64 from the run's binary32 values: l is the
// avoidance adjoint's result, returned is the λ before the move.
// An arrival's snap is constant under frozen decisions (λ = 0).  With carry,
// it is differentiated as if the arrival carried its leftover time onto the
// next road (nxt_tgt, nxt_road: the decisions after this tick),
// p' = T + (1 - L/s) s2 u2 with L = |T - p|, u2 the next road's direction and
// s, s2 the two roads' speeds: λ = (s2/s) u (u2·λ'), ∂/∂θ[road] += v L s2/s²
// (u2·λ'), ∂/∂θ[next road] += v (1 - L/s)(u2·λ').
// An agent's terms for the road it is on are summed in acc and added to
// gtheta where, going back in time, it leaves the road (its arrival, about one
// tick in 25; k_dflush for the first road): 800k agents, one atomic each per
// tick, took 40 us.
template <bool UNIFORM>
__device__ __forceinline__ double2 dmove_adj(const DiffMove& m, uint32_t k, uint8_t flag, double2 l) {
    if (flag & kDiffNoMove) {
        return l;
    }
    const float2 p = m.tp.pos[k];
    const float2 T = m.tp.tgt[k];
    const uint32_t r = m.tp.road[k];
    const float v = UNIFORM ? m.spd_const : m.spd[k];
    const double s = static_cast<double>(v * m.theta[r]);  // the run's binary32 speed
    const double dx = static_cast<double>(T.x) - p.x;
    const double dy = static_cast<double>(T.y) - p.y;
    const double len = sqrt(dx * dx + dy * dy);
    if (flag & kDiffArrived) {
        double2 out = make_double2(0.0, 0.0);
        const uint32_t r2 = m.nxt_road[k];
        double on_next = m.acc[k], on_this = 0.0;
        if (m.carry) {
            const float2 T2 = m.nxt_tgt[k];
            const double ex = static_cast<double>(T2.x) - T.x;
            const double ey = static_cast<double>(T2.y) - T.y;
            const double E = sqrt(ex * ex + ey * ey);
            const double s2 = static_cast<double>(v * m.theta[r2]);
            // a zero speed (theta[r] == 0) carries nothing: the frozen snap
            if (E > 0.0 && s > 0.0) {
                const double ux = len > 0.0 ? dx / len : 0.0;
                const double uy = len > 0.0 ? dy / len : 0.0;
                const double g2 = (ex / E) * l.x + (ey / E) * l.y;
                out = make_double2(ux * (s2 / s) * g2, uy * (s2 / s) * g2);
                on_this = static_cast<double>(v) * (len * s2 / (s * s)) * g2;
                on_next += static_cast<double>(v) * (1.0 - len / s) * g2;
            }
        }
        m.acc[k] = on_this;
        if (on_next != 0.0) atomicAdd(&m.gtheta[r2], on_next);
        return out;
    }
    const double ux = dx / len;
    const double uy = dy / len;
    const double ul = ux * l.x + uy * l.y;
    const double f = s / len;
    m.acc[k] += static_cast<double>(v) * ul;
    return make_double2(l.x - f * (l.x - ux * ul), l.y - f * (l.y - uy * ul));
}

// One tick of the adjoint, lam -> lam_out in agent order.
// The first near_blocks workgroups take the avoidance over the tick's binning,
// in binary64 from the run's binary32 positions, for the listed slots, GROUPS
// groups each: lam + alpha * sum J dl at their agents, from there the move
// adjoint, and the alpha derivative sum lam . A.  The other workgroups take
// the move adjoint of the agents without neighbours.  (One launch: the second
// part fills what the first leaves idle, and lam is read once.  A gradient of
// 2 x 1.5k agents over 40 ticks 2.40 -> 2.35 ms, of 8 x 100k over 100 16.0 ->
// 15.0; the second part first: 2.44 and 16.5.)
// Without lists (alpha = 0: the forward run had no avoidance to list them in)
// the first part sums the derivative over all slots and the second takes all
// agents.
template <uint32_t GROUPS, bool UNIFORM>
static __global__ __launch_bounds__(kBlock) void k_dadjoint(DiffCells c, DiffNear near, double alpha,
                                                     uint32_t near_blocks, DiffMove mv,
                                                     const double2* __restrict__ lam,
                                                     double2* __restrict__ lam_out, double* __restrict__ galpha) {
    __shared__ double red[kBlock / 64];
    if (blockIdx.x >= near_blocks) {
        const uint32_t k = (blockIdx.x - near_blocks) * kBlock + threadIdx.x;
        if (k < mv.n) {
            const uint8_t flag = mv.tp.flag[k];
            if (!(flag & kDiffNear)) lam_out[k] = dmove_adj<UNIFORM>(mv, k, flag, lam[k]);
        }
        return;
    }
    const uint32_t blk = collide_order(blockIdx.x, near_blocks);
    const uint32_t n_groups = (c.n + kNearGroup - 1u) / kNearGroup, g0 = blk * GROUPS;
    uint32_t end[GROUPS];
    uint32_t m = 0;
#pragma unroll
    for (uint32_t k = 0; k < GROUPS; k++) {
        if (g0 + k < n_groups) {
            m += near.list ? near.count[g0 + k] : min(kNearGroup, c.n - (g0 + k) * kNearGroup);
        }
        end[k] = m;
    }
    double ga = 0.0;
    for (uint32_t e = threadIdx.x; e < m; e += kBlock) {
        uint32_t k = 0, first = 0;
#pragma unroll
        for (uint32_t u = 0; u + 1u < GROUPS; u++) {
            if (e >= end[u]) {
                k = u + 1u;
                first = end[u];
            }
        }
        const uint32_t base = (g0 + k) * kNearGroup;
        const uint32_t s = base + (near.list ? near.list[base + (e - first)] : e - first);
        const float2 me = c.bpos[s];
        const uint32_t i = c.bid[s];
        const double2 li = lam[i];
        const double inv_r2 = c.inv_r2_d;
        double gx = 0.0, gy = 0.0, ax = 0.0, ay = 0.0;
        auto add = [&](float2 q, double2 lj) {
            const double x = static_cast<double>(me.x) - q.x;
            const double y = static_cast<double>(me.y) - q.y;
            const double h = 1.0 - (x * x + y * y) * inv_r2;
            const double w = h * h * h;
            const double wp = -3.0 * inv_r2 * h * h;  // dw/dq
            const double dlx = li.x - lj.x;
            const double dly = li.y - lj.y;
            const double xd = 2.0 * wp * (x * dlx + y * dly);
            gx += w * dlx + xd * x;
            gy += w * dly + xd * y;
            ax += w * x;
            ay += w * y;
        };
        // neighbours wait in a queue, so that their loads go out together
        uint32_t queue[4] = {s, s, s, s}, waiting = 0;
        for_neighbours(c, s, me, [&](uint32_t k) {
            if (waiting == 4u) {
                add(c.bpos[queue[3]], lam[c.bid[queue[3]]]);
                waiting--;
            }
            queue[3] = queue[2];
            queue[2] = queue[1];
            queue[1] = queue[0];
            queue[0] = k;
            waiting++;
        });
        uint32_t id[4];
        float2 q[4];
        double2 lj[4];
#pragma unroll
        for (uint32_t k = 0; k < 4u; k++) {
            id[k] = c.bid[queue[k]];
            q[k] = c.bpos[queue[k]];
        }
#pragma unroll
        for (uint32_t k = 0; k < 4u; k++) lj[k] = lam[id[k]];
#pragma unroll
        for (uint32_t k = 0; k < 4u; k++) {
            if (waiting > k) add(q[k], lj[k]);
        }
        if (near.list) {
            lam_out[i] = dmove_adj<UNIFORM>(mv, i, mv.tp.flag[i],
                                            make_double2(li.x + alpha * gx, li.y + alpha * gy));
        }
        ga += li.x * ax + li.y * ay;
    }
    if (m == 0u) {
        return;  // workgroup-uniform
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        ga += __shfl_xor(ga, o, 64);
    }
    if (__lane_id() == 0) red[threadIdx.x >> 6] = ga;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
#pragma unroll
        for (uint32_t k = 0; k < kBlock / 64; k++) t += red[k];
        if (t != 0.0) atomicAdd(&galpha[(blk % kAlphaSlots) * kAlphaStride], t);
    }
}

// The sums of the roads the agents start on, and the alpha derivative.
static __global__ __launch_bounds__(kBlock) void k_dflush(uint32_t n, const uint32_t* __restrict__ road,
                                                   const double* __restrict__ acc, double* __restrict__ gtheta,
                                                   const double* __restrict__ alpha_slots,
                                                   double* __restrict__ galpha) {
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k < n && acc[k] != 0.0) atomicAdd(&gtheta[road[k]], acc[k]);
    if (blockIdx.x == 0 && threadIdx.x < 64u) {
        static_assert(kAlphaSlots == 64u, "one wave sums the slots");
        double v = alpha_slots[threadIdx.x * kAlphaStride];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            v += __shfl_xor(v, o, 64);
        }
        if (threadIdx.x == 0) *galpha = v;
    }
}

// Caller order <-> internal order (perm: internal slot -> caller index).
static __global__ __launch_bounds__(kBlock) void k_dscatter(uint32_t n, const uint32_t* __restrict__ perm,
                                                     const float2* __restrict__ in, float2* __restrict__ out) {
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k < n) out[perm[k]] = in[k];
}

// The adjoint's start: the caller's gradient in agent order, the sums cleared.
static __global__ __launch_bounds__(kBlock) void k_dgather(uint32_t n, const uint32_t* __restrict__ perm,
                                                    const float2* __restrict__ in, double2* __restrict__ out,
                                                    double* __restrict__ acc, uint32_t n_roads,
                                                    double* __restrict__ gtheta, double* __restrict__ alpha_slots) {
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    for (uint32_t r = k; r < n_roads; r += gridDim.x * kBlock) gtheta[r] = 0.0;
    for (uint32_t w = k; w < kAlphaSlots * kAlphaStride; w += gridDim.x * kBlock) alpha_slots[w] = 0.0;
    if (k < n) {
        const float2 v = in[perm[k]];
        out[k] = make_double2(v.x, v.y);
        acc[k] = 0.0;
    }
}

// The parameters of a run are checked, and its window margins made, on the
// device: the host needs only the verdict.  (Read back, checked and uploaded
// again by the host, at the start of the forward and of the backward run: a
// gradient of 8 x 100k agents on 268k roads and 100 ticks took 16.8 ms, now
// 16.0; a run of 350k agents on 117k roads and 150 ticks 6.19, now 6.02.)
struct ParamWords {
    uint32_t most;  // bits of the largest multiplier
    uint32_t bad;   // one is negative, infinite or not a number
};

static __global__ __launch_bounds__(kBlock) void k_dcheck(const float* __restrict__ theta, uint32_t n,
                                                          ParamWords* __restrict__ words) {
    __shared__ float wave_most[kBlock / 64];
    float mx = 0.0f;
    bool bad = false;
#pragma unroll 4
    for (uint32_t r = blockIdx.x * kBlock + threadIdx.x; r < n; r += gridDim.x * kBlock) {
        const float t = theta[r];
        bad = bad || !(t >= 0.0f) || t > 3.402823466e38f;
        mx = t > mx ? t : mx;
    }
    for (uint32_t off = 32u; off > 0u; off >>= 1) {
        const float o = __shfl_xor(mx, off);
        mx = o > mx ? o : mx;
    }
    const bool any = __syncthreads_or(bad) != 0;
    if (__lane_id() == 0u) wave_most[threadIdx.x / 64u] = mx;
    __syncthreads();
    if (threadIdx.x == 0u) {
        for (uint32_t w = 1; w < kBlock / 64u; w++) mx = wave_most[w] > mx ? wave_most[w] : mx;
        if (mx > 0.0f) atomicMax(&words->most, __float_as_uint(mx));  // bits of floats >= 0 order as they do
        if (any) atomicOr(&words->bad, 1u);
    }
}

// Unless a multiplier is bad: theta into dst (if not there) and the margins of
// the scenario tables, (D + 1) rows and D columns for displacements of up to
// smax * theta + push.  next: the words of the next check, cleared.
static __global__ __launch_bounds__(kBlock) void k_dparams(const float* theta, float* dst, uint32_t n,
                                                           const ParamWords* __restrict__ words,
                                                           ParamWords* __restrict__ next, ScenDev* __restrict__ scen,
                                                           uint32_t n_scen, double smax, double push, double cell,
                                                           Mailbox* box, unsigned int report) {
    const bool bad = words->bad != 0u;
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (!bad) {
        if (dst != theta) {
            for (uint32_t r = k; r < n; r += gridDim.x * kBlock) dst[r] = theta[r];
        }
        const double disp = __dadd_rn(__dmul_rn(smax, static_cast<double>(__uint_as_float(words->most))), push);
        const double cells = floor(__dmul_rn(disp, 1.0 + 1.0 / 1048576.0) / cell);
        // beyond 64 bits: any number (such a run ends in kFaultBinCount)
        const uint32_t D = (cells < 9.0e18 ? static_cast<uint32_t>(static_cast<long long>(cells)) : 0u) + 1u;
        for (uint32_t i = k; i < n_scen; i += gridDim.x * kBlock) {
            scen[i].margin = (D + 1u) * (scen[i].wmask + 1u) + D;
        }
    }
    if (k == 0u) {
        *next = ParamWords{0u, 0u};
        __hip_atomic_store(&box->word, static_cast<unsigned long long>(report) << 32 | (bad ? 1u : 0u),
                           __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

}  // namespace msim

// ---------------------------------------------------------------------------

struct DiffSnapshot {
    uint32_t* perm = nullptr;  // initial snapshot only: agent order and speeds
    float* spd = nullptr;
    float2* pos = nullptr;
    float2* tgt = nullptr;
    uint32_t* road = nullptr;
    uint4* rng = nullptr;
    uint32_t* start = nullptr;
    uint32_t* bid = nullptr;
    float2* bpos = nullptr;
};

struct DiffState {
    uint32_t T = 0, C = 50, n_ck = 0;
    bool keep_schedule = false;
    bool no_move_first = false;
    bool carry = false;  // arrivals differentiated as carrying their leftover time
    bool have_forward = false;
    float alpha = 0.0f;      // parameters of the last recorded forward run
    float* theta = nullptr;  // [n_roads]
    float alpha_rep = 0.0f;  // parameters of the last replay
    float* theta_rep = nullptr;
    DiffSnapshot init;
    std::vector<DiffSnapshot> ck;
    // per-tick tape of one segment (or of the whole run with keep_schedule)
    DiffTapeDev tape{};      // [C][n] each
    uint32_t* tp_start = nullptr;  // [C][start_len]
    uint32_t* tp_bid = nullptr;    // [C][n]
    float2* tp_bpos = nullptr;     // [C][n + 2]
    uint8_t* tp_near = nullptr;    // [C][near_bytes(n)] lists and counts of the slots with neighbours
    // the tape holds the last segment of the latest forward run (recorded as
    // it ran, so that the backward pass need not replay it)
    bool tape_is_last = false;
    DiffTapeDev sched{};     // [T + 1][n] decisions of the whole run and those after it (keep_schedule)
    double2* lam = nullptr;  // adjoint state, agent order
    double2* lam2 = nullptr;
    double* acc = nullptr;   // [n] theta terms of the road each agent is on
    double* gtheta = nullptr;
    double* galpha = nullptr;
    double* alpha_slots = nullptr;  // [kAlphaSlots * kAlphaStride]
    ScenDev* scen = nullptr;  // scenario tables with the differentiable tick's margins
    ParamWords* words = nullptr;   // [2], one check's while the other's are cleared
    unsigned int checks = 0;
    float smax = 0.0f;  // largest base speed
    uint32_t max_block = 1;  // most agents in one 3x3 cell block of the initial binning
    float push_allow = 0.0f;  // avoidance push per axis the window margins allow for
    uint64_t generation = 0;  // recorded (non-replay) forward runs so far
};

namespace {

DiffTapeDev tape_at(const DiffTapeDev& t, size_t n, uint32_t k) {
    return DiffTapeDev{t.pos + n * k, t.tgt + n * k, t.road + n * k, t.flag + n * k};
}

size_t near_groups(uint32_t n) { return (static_cast<size_t>(n) + kNearGroup - 1) / kNearGroup; }
size_t near_bytes(uint32_t n) { return near_groups(n) * (kNearGroup + 1); }

// Tape entry k's neighbour lists.
DiffNear near_at(const msim_batch* b, const DiffState& d, uint32_t k) {
    uint8_t* p = d.tp_near + near_bytes(b->n) * k;
    return DiffNear{p, p + near_groups(b->n) * kNearGroup, d.tape.flag + static_cast<size_t>(b->n) * k};
}

int alloc_snapshot(msim_batch* b, DiffSnapshot& s) {
    int rc = balloc_n(b, &s.pos, b->n);
    if (rc == MSIM_OK) rc = balloc_n(b, &s.tgt, b->n);
    if (rc == MSIM_OK) rc = balloc_n(b, &s.road, b->n);
    if (rc == MSIM_OK) rc = balloc_n(b, &s.rng, b->n);
    if (rc == MSIM_OK) rc = balloc_n(b, &s.start, b->start_len);
    if (rc == MSIM_OK) rc = balloc_n(b, &s.bid, b->n);
    if (rc == MSIM_OK) rc = balloc_n(b, &s.bpos, static_cast<size_t>(b->n) + 2);
    return rc;
}

template <class T>
void dcopy(msim_batch* b, T* dst, const T* src, size_t count) {
    if (count) (void)hipMemcpyAsync(dst, src, count * sizeof(T), hipMemcpyDeviceToDevice, b->stream);
}

// The arrays of a snapshot, copied in one launch (k_copy_parts).
struct Copies {
    CopyParts p{};
    uint32_t parts = 0;
    size_t most = 0;
    template <class T>
    void add(T* dst, const T* src, size_t count) {
        if (!count) return;
        p.src[parts] = reinterpret_cast<const uint32_t*>(src);
        p.dst[parts] = reinterpret_cast<uint32_t*>(dst);
        p.words[parts++] = count * (sizeof(T) / 4);
        most = std::max(most, count * (sizeof(T) / 4));
    }
    void launch(msim_batch* b) const {
        if (!parts) return;
        const size_t blocks = (most + kCopyWords - 1) / kCopyWords;
        hipLaunchKernelGGL(k_copy_parts, dim3(static_cast<uint32_t>(std::min<size_t>(blocks, kCopyBlocks)), parts),
                           dim3(kBlock), 0, b->stream, p);
    }
};

// Working agent state (buffer cur) and the current binning (bcur) <-> snapshot.
void save_snapshot(msim_batch* b, DiffSnapshot& s) {
    const BBuffers& w = b->buf[b->cur];
    Copies c;
    c.add(s.pos, w.pos, b->n);
    c.add(s.tgt, w.tgt, b->n);
    c.add(s.road, w.road, b->n);
    c.add(s.rng, w.rng, b->n);
    c.add(s.start, b->bstart[b->bcur], b->start_len);
    c.add(s.bid, b->bbid[b->bcur], b->n);
    c.add(s.bpos, b->bbpos[b->bcur], b->n);
    c.launch(b);
}

void add_agents(msim_batch* b, Copies& c, const DiffSnapshot& s) {
    const BBuffers& w = b->buf[b->cur];
    c.add(w.pos, s.pos, b->n);
    c.add(w.tgt, s.tgt, b->n);
    c.add(w.road, s.road, b->n);
    c.add(w.rng, s.rng, b->n);
}

void load_agents(msim_batch* b, const DiffSnapshot& s) {
    Copies c;
    add_agents(b, c, s);
    c.launch(b);
}

// The initial state: agent order, speeds, agent state and binning.
void load_initial(msim_batch* b, const DiffSnapshot& s) {
    const BBuffers& w = b->buf[b->cur];
    Copies c;
    c.add(w.perm, s.perm, b->n);
    if (!b->uniform) c.add(w.spd, s.spd, b->n);
    add_agents(b, c, s);
    c.add(b->bstart[b->bcur], s.start, b->start_len);
    c.add(b->bbid[b->bcur], s.bid, b->n);
    c.add(b->bbpos[b->bcur], s.bpos, b->n);
    c.launch(b);
}

// Largest push per axis of a differentiable tick that the rebinning windows
// allow for (the margins: speed * largest multiplier + push, k_dparams).
// The push is |alpha| sum_j w x_j <= |alpha| k max_u (1 - u^2)^3 u R
// (u = |x| / R; the maximum, at u^2 = 1/7, is below 0.24) for k neighbours;
// the windows allow for k = the most agents found in one 3x3 block of cells
// at set-up, and at least 2R.  A larger push (agents bunched tighter later)
// is caught on the device (kFaultBinCount, the run fails).
double diff_push(const msim_batch* b, const DiffState& d, float alpha) {
    return std::max(2.0 * b->radius, 0.24 * std::fabs(static_cast<double>(alpha)) * d.max_block *
                                         static_cast<double>(b->radius));
}

// Rebinning of the working positions: old binning -> new binning.
void dbins(msim_batch* b, const DiffState& d, const uint32_t* old_start, const uint32_t* old_bid,
           uint32_t* new_start, float2* new_bpos, uint32_t* new_bid) {
    BatchBin bb{};
    bb.scen = d.scen;
    bb.seg_scen = b->seg_scen;
    bb.old_start = old_start;
    bb.old_bid = old_bid;
    bb.new_start = new_start;
    bb.new_bpos = new_bpos;
    bb.new_bid = new_bid;
    bb.seg_total = b->seg_total;
    bb.faults = b->faults;
    bb.inv_cell = b->inv_cell;
    const size_t lds = sizeof(uint32_t) << b->max_seg_log;
    const float2* pos = b->buf[b->cur].pos;
    hipLaunchKernelGGL((k_bbin_count<4, kBinThreads>), dim3(b->n_seg), dim3(kBinThreads), lds, b->stream, pos, bb);
    hipLaunchKernelGGL((k_bbin_place<4, kBinThreads>), dim3(b->n_seg), dim3(kBinThreads), lds, b->stream, pos, bb);
}

DiffCells dcells(msim_batch* b, const uint32_t* start, const float2* bpos, const uint32_t* bid) {
    DiffCells c{};
    c.blk = b->blk_scen;
    c.scen = b->scen;
    c.agent_off = b->agent_off;
    c.n = b->n;
    c.start = start;
    c.bpos = bpos;
    c.bid = bid;
    c.inv_cell = b->inv_cell;
    c.d2_limit = b->d2_limit;
    c.inv_r2 = 1.0f / (b->radius * b->radius);
    c.inv_r2_d = 1.0 / (static_cast<double>(b->radius) * b->radius);
    // |w x| < R: terms below 2^40 units, sums of up to 2^22 terms in range
    c.fix_scale = std::ldexp(1.0f, 40 - std::max(0, static_cast<int>(std::ceil(std::log2(b->radius)))));
    c.push_allow = b->diff ? b->diff->push_allow : 0.0f;
    return c;
}

// One differentiable tick t on the working state: move (decide or replay),
// rebin into (start, bpos, bid), avoidance.
void dtick(msim_batch* b, DiffState& d, const float* theta, float alpha, uint32_t t, bool replay, DiffTapeDev rec,
           const uint32_t* old_start, const uint32_t* old_bid, uint32_t* new_start, float2* new_bpos,
           uint32_t* new_bid, DiffNear near = DiffNear{}) {
    const AgentsDev a = b->agents(b->cur);
    const uint32_t no_move = (t == 0 && d.no_move_first) ? 1u : 0u;
    const DiffTapeDev in = replay ? tape_at(d.sched, b->n, t) : DiffTapeDev{};
    const dim3 g(bblocks(b->n));
    if (replay) {
        if (b->uniform) {
            hipLaunchKernelGGL((k_dadvance<true, true>), g, dim3(kBlock), 0, b->stream, a, theta, no_move, in, rec,
                               b->roads, b->conns);
        } else {
            hipLaunchKernelGGL((k_dadvance<true, false>), g, dim3(kBlock), 0, b->stream, a, theta, no_move, in,
                               rec, b->roads, b->conns);
        }
    } else {
        if (b->uniform) {
            hipLaunchKernelGGL((k_dadvance<false, true>), g, dim3(kBlock), 0, b->stream, a, theta, no_move, in,
                               rec, b->roads, b->conns);
        } else {
            hipLaunchKernelGGL((k_dadvance<false, false>), g, dim3(kBlock), 0, b->stream, a, theta, no_move, in,
                               rec, b->roads, b->conns);
        }
    }
    dbins(b, d, old_start, old_bid, new_start, new_bpos, new_bid);
    if (alpha != 0.0f) {
        hipLaunchKernelGGL(k_davoid<1>, g, dim3(kBlock), 0, b->stream, dcells(b, new_start, new_bpos, new_bid),
                           alpha, a.pos, near, b->faults);
    }
}

// Tick t as entry j of the segment tape; the segment starts from (start, bid).
void dtick_taped(msim_batch* b, DiffState& d, uint32_t t, uint32_t j, const uint32_t* start, const uint32_t* bid) {
    const size_t n = b->n, m = b->start_len;
    dtick(b, d, d.theta, d.alpha, t, false, tape_at(d.tape, n, j), j ? d.tp_start + m * (j - 1) : start,
          j ? d.tp_bid + n * (j - 1) : bid, d.tp_start + m * j, d.tp_bpos + (n + 2) * j, d.tp_bid + n * j,
          near_at(b, d, j));
}

template <uint32_t GROUPS, bool UNIFORM>
void launch_dadjoint_g(msim_batch* b, const DiffState& d, const DiffCells& c, const DiffNear& near,
                       const DiffMove& mv) {
    constexpr uint32_t kSlotsPer = GROUPS * kNearGroup;
    const uint32_t nb = std::max(1u, (b->n + kSlotsPer - 1u) / kSlotsPer);
    hipLaunchKernelGGL((k_dadjoint<GROUPS, UNIFORM>), dim3(nb + bblocks(b->n)), dim3(kBlock), 0, b->stream, c, near,
                       static_cast<double>(d.alpha), nb, mv, d.lam, d.lam2, d.alpha_slots);
}

// The workgroups with the listed slots are the long ones: all of them start at
// once (five a CU) up to 640k agents, by taking more groups each.  Gradients
// over 30 ticks with 4, 8, 16 and 32 groups, us: 300k agents 2,127, 2,142,
// 2,208, 2,477; 600k 3,361, 3,071, 3,093, 3,467; 1.6M 7,142, 6,435, 6,220,
// 6,330; 3.2M 13,365, 11,862, 11,327, 11,292.  (Six workgroups a CU, by
// spilling: 800k agents over 100 ticks 14.9 -> 15.2 ms.)
template <bool UNIFORM>
void launch_dadjoint(msim_batch* b, const DiffState& d, const DiffCells& c, const DiffNear& near, const DiffMove& mv) {
    constexpr uint32_t kAtOnce = 5u * kCus;
    if (b->n <= kAtOnce * 4u * kNearGroup) {
        launch_dadjoint_g<4, UNIFORM>(b, d, c, near, mv);
    } else if (b->n <= kAtOnce * 8u * kNearGroup) {
        launch_dadjoint_g<8, UNIFORM>(b, d, c, near, mv);
    } else {
        launch_dadjoint_g<16, UNIFORM>(b, d, c, near, mv);
    }
}

int check_diff_faults(msim_batch* b) {
    unsigned int f = 0;
    int rc = bwait_report(b, &f);
    if (rc != MSIM_OK) return rc;
    if (f & kFaultBinCount) {
        return bfail(b, MSIM_ERR_STATE,
                     "an agent moved beyond its rebinning window in a differentiable tick (theta or alpha too "
                     "large for the window margins)");
    }
    if (f) return bfail(b, MSIM_ERR_STATE, "device-side check failed (fault bits 0x%x)", f);
    return MSIM_OK;
}

}  // namespace

void diff_release(msim_batch* b) {
    delete b->diff;  // device memory is in b->allocs
    b->diff = nullptr;
}

extern "C" int msim_batch_diff_setup(msim_batch* b, uint32_t n_ticks, uint32_t checkpoint_every,
                                     int keep_schedule) {
    if (!b) return bfail(b, MSIM_ERR_INVALID, "NULL handle");
    if (b->diff) return bfail(b, MSIM_ERR_STATE, "the differentiable tick is already set up on this handle");
    if (n_ticks == 0 || checkpoint_every == 0) return bfail(b, MSIM_ERR_INVALID, "n_ticks and checkpoint_every must be > 0");
    int rc = bleave_sorted(b);  // the differentiable tick runs on the classic layout
    if (rc == MSIM_OK) rc = msim_batch_sync(b);
    if (rc != MSIM_OK) return rc;
    DiffState* d = new DiffState();
    b->diff = d;
    const DeviceScope scope(b->device);  // copies below run on its null stream
    d->T = n_ticks;
    d->C = std::min(checkpoint_every, n_ticks);
    d->n_ck = (n_ticks + d->C - 1) / d->C;
    d->keep_schedule = keep_schedule != 0;
    d->no_move_first = b->first_tick_insert_only;
    const size_t n = b->n;
    rc = balloc_n(b, &d->theta, b->n_roads);
    if (rc == MSIM_OK) rc = balloc_n(b, &d->theta_rep, b->n_roads);
    if (rc == MSIM_OK) rc = alloc_snapshot(b, d->init);
    if (rc == MSIM_OK) rc = balloc_n(b, &d->init.perm, n);
    if (rc == MSIM_OK && !b->uniform) rc = balloc_n(b, &d->init.spd, n);
    d->ck.resize(d->n_ck);
    for (uint32_t k = 0; k < d->n_ck && rc == MSIM_OK; k++) rc = alloc_snapshot(b, d->ck[k]);
    if (rc == MSIM_OK) rc = balloc_n(b, &d->tape.pos, n * d->C);
    if (rc == MSIM_OK) rc = balloc_n(b, &d->tape.tgt, n * d->C);
    if (rc == MSIM_OK) rc = balloc_n(b, &d->tape.road, n * d->C);
    if (rc == MSIM_OK) rc = balloc_n(b, &d->tape.flag, n * d->C);
    if (rc == MSIM_OK) rc = balloc_n(b, &d->tp_start, static_cast<size_t>(b->start_len) * d->C);
    if (rc == MSIM_OK) rc = balloc_n(b, &d->tp_bid, n * d->C);
    if (rc == MSIM_OK) rc = balloc_n(b, &d->tp_bpos, (n + 2) * d->C);
    if (rc == MSIM_OK) rc = balloc_n(b, &d->tp_near, near_bytes(b->n) * d->C);
    if (rc == MSIM_OK && d->keep_schedule) {
        rc = balloc_n(b, &d->sched.pos, n * (n_ticks + 1u));
        if (rc == MSIM_OK) rc = balloc_n(b, &d->sched.tgt, n * (n_ticks + 1u));
        if (rc == MSIM_OK) rc = balloc_n(b, &d->sched.road, n * (n_ticks + 1u));
        if (rc == MSIM_OK) rc = balloc_n(b, &d->sched.flag, n * (n_ticks + 1u));
    }
    if (rc == MSIM_OK) rc = balloc_n(b, &d->lam, n);
    if (rc == MSIM_OK) rc = balloc_n(b, &d->lam2, n);
    if (rc == MSIM_OK) rc = balloc_n(b, &d->gtheta, b->n_roads);
    if (rc == MSIM_OK) rc = balloc_n(b, &d->galpha, 1);
    if (rc == MSIM_OK) rc = balloc_n(b, &d->acc, n);
    if (rc == MSIM_OK) rc = balloc_n(b, &d->alpha_slots, kAlphaSlots * kAlphaStride);
    if (rc == MSIM_OK) rc = balloc_n(b, &d->scen, b->n_scen);
    if (rc == MSIM_OK) rc = balloc_n(b, &d->words, 2);
    std::vector<ScenDev> scen_h(b->n_scen);
    if (rc == MSIM_OK) {
        b->verdict->word = 0;
        const ParamWords none[2] = {};
        hipError_t e = hipMemcpy(d->words, none, sizeof(none), hipMemcpyHostToDevice);
        if (e == hipSuccess) {
            e = hipMemcpy(scen_h.data(), b->scen, sizeof(ScenDev) * b->n_scen, hipMemcpyDeviceToHost);
        }
        if (e == hipSuccess) e = hipMemcpy(d->scen, b->scen, sizeof(ScenDev) * b->n_scen, hipMemcpyDeviceToDevice);
        if (e == hipSuccess) e = wait_null_stream(b->device);
        if (e != hipSuccess) rc = bfail(b, MSIM_ERR_HIP, "scenario table copy: %s", hipGetErrorString(e));
    }
    if (rc == MSIM_OK && b->start_len) {
        // the push allowance: at most 9 x the fullest bucket in a 3x3 block
        std::vector<uint32_t> st(b->start_len);
        hipError_t e = hipMemcpy(st.data(), b->bstart[b->bcur], sizeof(uint32_t) * b->start_len,
                                 hipMemcpyDeviceToHost);
        if (e != hipSuccess) rc = bfail(b, MSIM_ERR_HIP, "binning readback: %s", hipGetErrorString(e));
        uint32_t most = 1;
        for (const ScenDev& sc : scen_h) {
            for (uint32_t j = 0; j < sc.m && rc == MSIM_OK; j++) {
                most = std::max(most, st[sc.start_base + j + 1] - st[sc.start_base + j]);
            }
        }
        d->max_block = 9u * most;
    }
    if (rc == MSIM_OK) {
        d->smax = kShaderSpeed;
        if (!b->uniform) {
            std::vector<float> v(n);
            hipError_t e = n ? hipMemcpy(v.data(), b->buf[b->cur].spd, sizeof(float) * n, hipMemcpyDeviceToHost)
                             : hipSuccess;
            if (e != hipSuccess) rc = bfail(b, MSIM_ERR_HIP, "speed readback: %s", hipGetErrorString(e));
            d->smax = 0.0f;
            for (float s : v) d->smax = std::max(d->smax, s);
        }
    }
    if (rc == MSIM_OK) {
        save_snapshot(b, d->init);
        dcopy(b, d->init.perm, b->buf[b->cur].perm, n);
        if (!b->uniform) dcopy(b, d->init.spd, b->buf[b->cur].spd, n);
        rc = bwait(b);
    }
    if (rc != MSIM_OK) diff_release(b);
    return rc;
}

namespace {

// theta on the host, checked.
int read_theta(msim_batch* b, const float* theta, std::vector<float>& th) {
    th.resize(b->n_roads);
    if (b->n_roads) {
        hipError_t e = hipMemcpy(th.data(), theta, sizeof(float) * b->n_roads, hipMemcpyDeviceToHost);
        if (e != hipSuccess) return bfail(b, MSIM_ERR_HIP, "theta readback: %s", hipGetErrorString(e));
    }
    for (uint32_t r = 0; r < b->n_roads; r++) {
        if (!(th[r] >= 0.0f) || !std::isfinite(th[r])) {
            return bfail(b, MSIM_ERR_INVALID, "theta[%u] = %g is not a finite non-negative multiplier", r,
                         static_cast<double>(th[r]));
        }
    }
    return MSIM_OK;
}

// True: a kernel on the handle's device can read n floats there (memory of
// that device, aligned, as long as that).  Anything else goes through copies.
bool readable(const msim_batch* b, const float* p, size_t n) {
    hipPointerAttribute_t a{};
    hipDeviceptr_t base{};
    size_t size = 0;
    const uintptr_t at = reinterpret_cast<uintptr_t>(p);
    if (at % alignof(float) != 0 || hipPointerGetAttributes(&a, p) != hipSuccess || a.type != hipMemoryTypeDevice ||
        a.device != b->device ||
        hipMemGetAddressRange(&base, &size, reinterpret_cast<hipDeviceptr_t>(const_cast<float*>(p))) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    const uintptr_t end = reinterpret_cast<uintptr_t>(base) + size;
    return at < end && n * sizeof(float) <= end - at;
}

// Parameters: theta (device, n_roads packed, >= 0 and finite) into dst,
// alpha; the window margins follow the largest multiplier.
int set_params(msim_batch* b, DiffState& d, const float* theta, float alpha, float* dst) {
    if (!theta) return bfail(b, MSIM_ERR_INVALID, "NULL theta");
    if (!std::isfinite(alpha)) return bfail(b, MSIM_ERR_INVALID, "alpha must be finite");
    const uint32_t n = b->n_roads;
    std::vector<float> th;
    const bool direct = theta == dst || n == 0 || readable(b, theta, n);
    if (!direct) {
        int rc = read_theta(b, theta, th);
        if (rc != MSIM_OK) return rc;
        hipError_t e = hipMemcpy(dst, th.data(), sizeof(float) * n, hipMemcpyHostToDevice);
        if (e != hipSuccess) return bfail(b, MSIM_ERR_HIP, "theta upload: %s", hipGetErrorString(e));
    }
    // theta may come from work on the null stream of its device
    if (wait_null_stream(b->device) != hipSuccess) return bfail(b, MSIM_ERR_HIP, "parameter upload failed");
    const float* src = direct ? theta : dst;
    const unsigned int report = ++d.checks;
    ParamWords* const words = d.words + report % 2u;
    const uint32_t blocks = std::min(bblocks(std::max(n, b->n_scen)), 2u * kCus);
    const double push = diff_push(b, d, alpha);
    hipLaunchKernelGGL(k_dcheck, dim3(blocks), dim3(kBlock), 0, b->stream, src, n, words);
    hipLaunchKernelGGL(k_dparams, dim3(blocks), dim3(kBlock), 0, b->stream, src, dst, n, words,
                       d.words + (report + 1u) % 2u, d.scen, b->n_scen, static_cast<double>(d.smax), push,
                       static_cast<double>(1.0f / b->inv_cell), b->verdict, report);
    int rc = bcheck(b, "parameter check");
    if (rc == MSIM_OK && !await_report(b->verdict, report)) rc = bwait(b);
    if (rc != MSIM_OK) return rc;
    const unsigned long long verdict = __atomic_load_n(&b->verdict->word, __ATOMIC_ACQUIRE);
    if (static_cast<unsigned int>(verdict >> 32) != report) return bfail(b, MSIM_ERR_HIP, "no parameter report");
    if (verdict & 1ull) {
        rc = read_theta(b, theta, th);  // which one
        return rc != MSIM_OK ? rc : bfail(b, MSIM_ERR_INVALID, "theta is not finite and non-negative");
    }
    d.push_allow = static_cast<float>(push);
    return MSIM_OK;
}

}  // namespace

extern "C" int msim_batch_diff_forward(msim_batch* b, const float* theta, float alpha, int replay,
                                       float* final_pos) {
    if (!b || !b->diff) return bfail(b, MSIM_ERR_STATE, "msim_batch_diff_setup first");
    DiffState& d = *b->diff;
    if (replay && !(d.keep_schedule && d.have_forward)) {
        return bfail(b, MSIM_ERR_STATE, "replay needs keep_schedule and a recorded forward run");
    }
    int rc = msim_batch_sync(b);
    if (rc != MSIM_OK) return rc;
    float* th = replay ? d.theta_rep : d.theta;
    rc = set_params(b, d, theta, alpha, th);
    if (rc != MSIM_OK) return rc;
    if (replay) {
        d.alpha_rep = alpha;
    } else {
        d.alpha = alpha;
        d.have_forward = false;
    }
    load_initial(b, d.init);
    d.tape_is_last = false;
    const uint32_t t_last = (d.n_ck - 1) * d.C;  // the last segment's first tick
    for (uint32_t t = 0; t < d.T && rc == MSIM_OK; t++) {
        if (!replay && t % d.C == 0) save_snapshot(b, d.ck[t / d.C]);
        if (!replay && !d.keep_schedule && t >= t_last) {
            // on the tape, binning included (the working one ends here)
            dtick_taped(b, d, t, t - t_last, b->bstart[b->bcur], b->bbid[b->bcur]);
            rc = bcheck(b, "differentiable tick");
            continue;
        }
        const DiffTapeDev rec = (!replay && d.keep_schedule) ? tape_at(d.sched, b->n, t) : DiffTapeDev{};
        const int nb = 1 - b->bcur;
        dtick(b, d, th, alpha, t, replay != 0, rec, b->bstart[b->bcur], b->bbid[b->bcur], b->bstart[nb],
              b->bbpos[nb], b->bbid[nb]);
        b->bcur = nb;
        rc = bcheck(b, "differentiable tick");
    }
    if (rc == MSIM_OK && !replay && d.keep_schedule && b->n) {
        // the decisions in force after the last tick (schedule entry T)
        const DiffTapeDev fin = tape_at(d.sched, b->n, d.T);
        const AgentsDev a = b->agents(b->cur);
        hipError_t e = hipMemcpyAsync(fin.pos, a.pos, sizeof(float2) * b->n, hipMemcpyDeviceToDevice, b->stream);
        if (e == hipSuccess) {
            e = hipMemcpyAsync(fin.tgt, a.tgt, sizeof(float2) * b->n, hipMemcpyDeviceToDevice, b->stream);
        }
        if (e == hipSuccess) {
            e = hipMemcpyAsync(fin.road, a.road, sizeof(uint32_t) * b->n, hipMemcpyDeviceToDevice, b->stream);
        }
        if (e == hipSuccess) e = hipMemsetAsync(fin.flag, 0, b->n, b->stream);
        if (e != hipSuccess) rc = bfail(b, MSIM_ERR_HIP, "schedule copy: %s", hipGetErrorString(e));
    }
    if (rc == MSIM_OK && final_pos) {
        hipLaunchKernelGGL(k_dscatter, dim3(bblocks(b->n)), dim3(kBlock), 0, b->stream, b->n, b->buf[b->cur].perm,
                           b->buf[b->cur].pos, reinterpret_cast<float2*>(final_pos));
        rc = bcheck(b, "k_dscatter");
    }
    if (rc == MSIM_OK) rc = check_diff_faults(b);
    if (rc == MSIM_OK && !replay) {
        d.have_forward = true;
        d.tape_is_last = !d.keep_schedule;
        d.generation++;
    }
    return rc;
}

extern "C" int msim_batch_diff_generation(msim_batch* b, uint64_t* out) {
    if (!b || !b->diff || !out) return bfail(b, MSIM_ERR_STATE, "msim_batch_diff_setup first (or NULL argument)");
    *out = b->diff->generation;
    return MSIM_OK;
}

extern "C" int msim_batch_diff_backward(msim_batch* b, const float* grad_pos, double* grad_theta,
                                        double* grad_alpha) {
    if (!b || !b->diff) return bfail(b, MSIM_ERR_STATE, "msim_batch_diff_setup first");
    DiffState& d = *b->diff;
    if (!d.have_forward) return bfail(b, MSIM_ERR_STATE, "run msim_batch_diff_forward (not a replay) first");
    if (!grad_pos || !grad_theta || !grad_alpha) return bfail(b, MSIM_ERR_INVALID, "NULL argument");
    int rc = msim_batch_sync(b);
    if (rc != MSIM_OK) return rc;
    rc = set_params(b, d, d.theta, d.alpha, d.theta);  // margins of the recorded run
    if (rc != MSIM_OK) return rc;
    const size_t n = b->n;
    const dim3 g(bblocks(b->n));
    const uint32_t* perm = b->buf[b->cur].perm;
    hipLaunchKernelGGL(k_dgather, g, dim3(kBlock), 0, b->stream, b->n, perm,
                       reinterpret_cast<const float2*>(grad_pos), d.lam, d.acc, b->n_roads, d.gtheta, d.alpha_slots);
    for (int seg = static_cast<int>(d.n_ck) - 1; seg >= 0 && rc == MSIM_OK; seg--) {
        const uint32_t t0 = static_cast<uint32_t>(seg) * d.C;
        const uint32_t t1 = std::min(d.T, t0 + d.C);
        if (!d.tape_is_last) {  // replay the segment from its checkpoint, recording the tape
            load_agents(b, d.ck[seg]);
            for (uint32_t t = t0; t < t1; t++) dtick_taped(b, d, t, t - t0, d.ck[seg].start, d.ck[seg].bid);
        }
        d.tape_is_last = false;
        rc = bcheck(b, "differentiable tick (segment replay)");
        // reverse through the segment
        for (uint32_t t = t1; t-- > t0 && rc == MSIM_OK;) {
            const uint32_t j = t - t0;
            const DiffCells c = dcells(b, d.tp_start + static_cast<size_t>(b->start_len) * j, d.tp_bpos + (n + 2) * j,
                                       d.tp_bid + n * j);
            const AgentsDev a = b->agents(b->cur);
            // the decisions after tick t: the tape's next entry, or after the
            // segment's last tick the agent state its replay ended in
            const float2* nt = t + 1 < t1 ? tape_at(d.tape, n, j + 1).tgt : a.tgt;
            const uint32_t* nr = t + 1 < t1 ? tape_at(d.tape, n, j + 1).road : a.road;
            const DiffMove mv{b->n, a.spd, a.spd_const, d.theta, tape_at(d.tape, n, j), nt, nr, d.carry ? 1u : 0u,
                              d.acc, d.gtheta};
            const DiffNear near = d.alpha != 0.0f ? near_at(b, d, j) : DiffNear{};
            if (b->uniform) {
                launch_dadjoint<true>(b, d, c, near, mv);
            } else {
                launch_dadjoint<false>(b, d, c, near, mv);
            }
            std::swap(d.lam, d.lam2);
            rc = bcheck(b, "adjoint tick");
        }
    }
    if (rc == MSIM_OK) {
        // the tape's first entry is the run's first tick now
        hipLaunchKernelGGL(k_dflush, g, dim3(kBlock), 0, b->stream, b->n, d.tape.road, d.acc, d.gtheta,
                           d.alpha_slots, d.galpha);
        dcopy(b, grad_theta, d.gtheta, b->n_roads);
        dcopy(b, grad_alpha, d.galpha, 1);
        rc = check_diff_faults(b);
    }
    return rc;
}

extern "C" int msim_batch_diff_set_arrival_gradient(msim_batch* b, int mode) {
    if (!b || !b->diff) return bfail(b, MSIM_ERR_STATE, "msim_batch_diff_setup first");
    if (mode != 0 && mode != 1) return bfail(b, MSIM_ERR_INVALID, "arrival gradient mode must be 0 or 1");
    b->diff->carry = mode == 1;
    return MSIM_OK;
}

extern "C" int msim_batch_diff_read_schedule(msim_batch* b, uint32_t tick, float* target, uint32_t* road,
                                             uint8_t* flag) {
    if (!b || !b->diff) return bfail(b, MSIM_ERR_STATE, "msim_batch_diff_setup first");
    DiffState& d = *b->diff;
    if (!(d.keep_schedule && d.have_forward)) return bfail(b, MSIM_ERR_STATE, "no recorded schedule");
    if (tick > d.T) return bfail(b, MSIM_ERR_INVALID, "tick %u beyond the run's %u ticks", tick, d.T);
    int rc = msim_batch_sync(b);
    if (rc != MSIM_OK) return rc;
    const size_t n = b->n;
    std::vector<float2> t(n);
    std::vector<uint32_t> r(n), perm(n);
    std::vector<uint8_t> f(n);
    const DiffTapeDev s = tape_at(d.sched, n, tick);
    hipError_t e = hipSuccess;
    if (n) {
        e = hipMemcpy(t.data(), s.tgt, sizeof(float2) * n, hipMemcpyDeviceToHost);
        if (e == hipSuccess) e = hipMemcpy(r.data(), s.road, sizeof(uint32_t) * n, hipMemcpyDeviceToHost);
        if (e == hipSuccess) e = hipMemcpy(f.data(), s.flag, n, hipMemcpyDeviceToHost);
        if (e == hipSuccess) e = hipMemcpy(perm.data(), b->buf[b->cur].perm, sizeof(uint32_t) * n, hipMemcpyDeviceToHost);
    }
    if (e != hipSuccess) return bfail(b, MSIM_ERR_HIP, "schedule readback: %s", hipGetErrorString(e));
    for (size_t k = 0; k < n; k++) {
        const uint32_t i = perm[k];
        if (target) {
            target[2 * i] = t[k].x;
            target[2 * i + 1] = t[k].y;
        }
        if (road) road[i] = r[k];
        if (flag) flag[i] = f[k];
    }
    return MSIM_OK;
}
