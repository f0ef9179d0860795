// Persistent lane-refill work loop for wave64.
//
// The Mandelbulb iteration count varies wildly between neighbouring points
// (on the 64^3 grid 73% of points bail after one body and 8% run all 15), so
// a wave that gives each lane one point idles most lanes while its slowest
// point finishes.  Here every lane owns one point at a time; when its point
// finishes (bailout or iteration cap) the lane writes the result and takes
// the next index from the wave's chunk, so all lanes keep executing loop
// bodies.  Chunks of `chunk` consecutive indices are dealt to the waves: the
// first of every wave by its number, further ones either by number as well
// (static) or from sharded counters with one atomic per wave (dynamic).  The
// last wave of a shard to leave resets its counter, so a launch leaves them
// at zero (safe for graph replay).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "de_device.h"

namespace cth {

struct WorkQueue {
    uint32_t* ctr;     // shard s: ctr[s * kShardStride] chunks claimed, [.. + 1] waves that have left
    uint32_t shards;   // a power of two (dynamic only)
    uint32_t waves;    // waves in the launch
    uint32_t total;    // indices in [0, total)
    uint32_t chunk;    // indices per chunk
    uint32_t chunks;   // ceil(total / chunk)
    uint32_t rotate;   // a wave's step from row to row of `waves` chunks (static), below `waves`
    uint32_t refill_min;  // idle lanes that trigger a write-back + refill (1..64)
    uint32_t dynamic;     // 1: claim chunks after the first with an atomic; 0: static interleave
    // Work counters (nullable): the launch adds its loop bodies, its
    // evaluations that ended by bailout, and its evaluations to
    // stats[0], stats[1], stats[2] (the counting instantiations only).
    unsigned long long* stats;
};

// Per-wave work tally of a refill kernel (wave-uniform, scalar registers):
// lane masks of the lanes that ran a loop body, that ended an evaluation by
// bailout, that started an evaluation.  Only the counting instantiation of a
// kernel (kOn, launched while a context counts work) tallies: even scalar
// adds in the tick cost measurable time (11% on the span kernel), and the
// counts depend only on the inputs, not on which instantiation ran.
template <bool kOn>
struct WorkTally {
    uint64_t bodies = 0, bails = 0, evals = 0;
    __device__ __forceinline__ void body(uint64_t m) {
        if constexpr (kOn) bodies += (uint64_t)__popcll(m);
    }
    __device__ __forceinline__ void bail(uint64_t m) {
        if constexpr (kOn) bails += (uint64_t)__popcll(m);
    }
    __device__ __forceinline__ void eval(uint64_t m) {
        if constexpr (kOn) evals += (uint64_t)__popcll(m);
    }
    __device__ __forceinline__ void flush(unsigned long long* stats) const {
        if constexpr (kOn) {
            if (!stats) return;
            const uint64_t active = wave_mask(true);
            if ((int)__lane_id() == __ffsll((unsigned long long)active) - 1) {
                atomicAdd(stats, (unsigned long long)bodies);
                atomicAdd(stats + 1, (unsigned long long)bails);
                atomicAdd(stats + 2, (unsigned long long)evals);
            }
        }
    }
};

__device__ __forceinline__ uint32_t lane_rank(uint64_t mask) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// The wave's LDS writes become visible to its other lanes.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One atomic per wave; the value is broadcast from the first active lane.
__device__ __forceinline__ uint32_t wave_claim(uint32_t* ctr, uint32_t amount) {
    uint64_t active = wave_mask(1);
    int leader = __ffsll((unsigned long long)active) - 1;
    uint32_t v = 0;
    if ((int)__lane_id() == leader) v = atomicAdd(ctr, amount);
    return (uint32_t)__builtin_amdgcn_readlane((int)v, leader);
}

// Wave index within the launch (read from the first lane so that the compiler
// knows it is wave-uniform and keeps the chunk window in scalar registers).
__device__ __forceinline__ uint32_t wave_id() {
    return blockIdx.x * (blockDim.x >> 6) + (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
}

constexpr uint32_t kNoChunk = ~0u;

// The wave's window of claimed indices (wave-uniform, scalar registers).
struct Window {
    uint32_t next = 0, end = 0;  // indices not handed out yet
    uint32_t row = 0;            // first chunk of the row of `waves` chunks it takes one of (static)
    uint32_t pos = kNoChunk;     // its place in that row; kNoChunk before the first chunk
    bool last = false;           // no chunk follows the current one
    // Idle lanes that trigger the wave's next refill: refill_min, or as few as
    // take the whole rest of the wave's last chunk, or, with no index left, the
    // whole wave (a batch that could not take new points is only written).
    __device__ __forceinline__ uint32_t refill_at(const WorkQueue& q) const {
        if (!last) return q.refill_min;
        return next >= end ? 64u : (end - next < q.refill_min ? end - next : q.refill_min);
    }
};

// The next chunk of the wave; false when the index space is exhausted.
// Chunk w goes to wave w first, so that a launch starts without claims and one
// that has no more chunks than waves makes none.  Further chunks are, static,
// one of each further row of W chunks (W waves: every wave is spread over the
// whole domain, so that slow and fast regions average out; its place moves by
// `rotate` from row to row, so that a row length that fits the domain, 4096
// waves of 256 indices in 128^3 grids, does not give a wave the same region
// every time); dynamic, the next unclaimed chunk of the workgroup's shard.
// Claims on one counter serialise at about 14 ns each, whatever the number of
// waves (17.6 M corners in 68,600 chunks of 256 took 971 us, and 137 us with 32
// shards), hence the shards: row j of the remaining chunks holds one for each
// shard, rotated from row to row so that no shard gets the same region of a
// regular index space every time.
__device__ __forceinline__ bool next_chunk(const WorkQueue& q, Window& w) {
    if (w.last) return false;
    uint32_t c;
    if (w.pos == kNoChunk) {
        w.pos = c = wave_id();
    } else if (!q.dynamic) {
        w.row += q.waves;
        w.pos += q.rotate;
        if (w.pos >= q.waves) w.pos -= q.waves;
        c = w.row + w.pos;
    } else {
        const uint32_t s = blockIdx.x & (q.shards - 1u);
        const uint32_t j = wave_claim(q.ctr + s * kShardStride, 1u);
        c = q.waves + j * q.shards + ((s + 11u * j) & (q.shards - 1u));
    }
    w.last = c >= q.chunks;
    if (w.last) return false;
    w.next = c * q.chunk;
    w.end = (q.total - w.next < q.chunk) ? q.total : w.next + q.chunk;
    if (!q.dynamic) {
        uint32_t p = w.pos + q.rotate;
        if (p >= q.waves) p -= q.waves;
        w.last = w.row + q.waves + p >= q.chunks;
    }
    return true;
}

// Called once per wave of a dynamic launch after its last claim; the final
// wave of a shard zeroes its counters.  Every other wave of the shard has
// already made its final claim by then.
__device__ __forceinline__ void wave_retire(const WorkQueue& q) {
    const uint64_t active = wave_mask(1);
    const int leader = __ffsll((unsigned long long)active) - 1;
    if ((int)__lane_id() == leader) {
        const uint32_t s = blockIdx.x & (q.shards - 1u);
        const uint32_t blocks = (gridDim.x - s + q.shards - 1u) / q.shards;  // workgroups of the shard
        uint32_t* ctr = q.ctr + s * kShardStride;
        if (atomicAdd(ctr + 1, 1u) == blocks * (blockDim.x >> 6) - 1u) {
            atomicExch(ctr, 0u);
            atomicExch(ctr + 1, 0u);
        }
    }
}

// Drive evaluator `Ev` over the indices of `q`, reading points from `src`
// and writing results through `sink`.
//   src.get(i, x, y, z, power)
//   sink.put(i, d, iters, r, dr, ev)  (ev: the evaluator, for derivative sinks)
//
// Each tick runs one loop body on every lane (results committed where the
// lane's point is live).  A lane whose point finishes holds (r, dr) until at
// least `q.refill_min` lanes of the wave are idle; then the held points are
// written and the idle lanes take new indices.  Batching the refill keeps the
// per-tick control flow to a few scalar instructions.
//
// Which lanes are live or hold a finished point is kept in wave-uniform lane
// masks (scalar registers).  A compare's lane mask is free to combine with
// them, and the per-lane view is the same mask
// (__builtin_amdgcn_inverse_ballot_w64).  A point's body count is the wave's
// tick counter (scalar) minus the tick at which the lane took the point, so
// the iteration cap costs one compare per tick and no per-lane counter.
//
// Evaluators with Ev::kLastDr end a point that reaches the iteration cap
// after max_iters - 1 bodies: of its max_iters-th body only the dr update is
// live (Ev::last_dr), and it is applied when the point is written (`last_m`
// marks those lanes).  r is then the magnitude that body would have read,
// which is the magnitude the reference ends with.
template <class Ev, bool kCount, class Src, class Sink>
__device__ __forceinline__ void refill_loop(const Src& src, const MandelUniform& u, const Sink& sink,
                                            const WorkQueue& q) {
    Ev ev;
    const uint64_t wave = wave_mask(true);  // the wave's lanes
    uint64_t live_m = 0;  // lanes whose point needs another loop body
    uint64_t hold_m = 0;  // lanes holding a finished point not yet written
    uint64_t last_m = 0;  // held points whose last body's dr update is due (kLastDr)
    uint32_t tick = 0;    // loop bodies run by the wave
    uint32_t idx = 0;
    uint32_t t0 = 0;      // tick at which the lane took its point
    uint32_t kh = 0;      // body count of a held point (kept if the sink reads it)
    float r = idle_start(ev, u);
    Window win;
    WorkTally<kCount> tally;

    for (;;) {
        // Refill; again at once if every point taken bailed before its first body.
        do {
            if (__builtin_amdgcn_inverse_ballot_w64(hold_m)) {
                if constexpr (Ev::kLastDr) {
                    if (__builtin_amdgcn_inverse_ballot_w64(last_m)) ev.last_dr(r);
                }
                sink.put(idx, ev.finish(r), kh, r, ev.dr, ev);
            }
            hold_m = 0;
            last_m = 0;
            // Hand new points to idle lanes.  A point that bails before its
            // first body (|p| > bailout) is held like any finished one, until
            // the next refill; a few idle lanes that took a run of such points
            // in turn would hold up the wave (one lane, 64 points: 50 us of a
            // 96^3 grid's 66).
            uint64_t need = wave & ~live_m;
            while (need != 0) {
                if (win.next >= win.end && !next_chunk(q, win)) break;
                const uint32_t avail = win.end - win.next;
                const uint32_t nneed = (uint32_t)__popcll(need);
                const uint32_t rank = lane_rank(need);
                const bool take = __builtin_amdgcn_inverse_ballot_w64(need) && rank < avail;
                if (take) {
                    idx = win.next + rank;
                    float px, py, pz, pw;
                    src.get(idx, px, py, pz, pw);
                    ev.start(px, py, pz, pw, u);
                    t0 = tick;
                    r = ev.mag();
                }
                const uint64_t took = wave_mask(take);
                const uint64_t bailed = wave_mask(r > u.bailout) & took;
                tally.eval(took);
                tally.bail(bailed);
                // With kLastDr and max_iters == 1 a point that does not bail
                // at once is at its cap before any full body.
                const uint64_t capped = (Ev::kLastDr && u.max_iters == 1u) ? took & ~bailed : 0;
                tally.body(capped);
                last_m |= capped;
                hold_m |= bailed | capped;
                if (sink.wants_k() && (bailed | capped) != 0) {
                    if (__builtin_amdgcn_inverse_ballot_w64(bailed | capped))
                        kh = __builtin_amdgcn_inverse_ballot_w64(capped) ? 1u : 0u;
                }
                live_m |= took & ~(bailed | capped);
                need &= ~took;
                win.next += (nneed < avail) ? nneed : avail;
            }
        } while (live_m == 0 && hold_m != 0);
        if (live_m == 0) break;
        tick_guard(ev, u);  // the started points' squares
        // Idle lanes, win.refill_at() of them, trigger the next refill.
        const uint32_t limit = 64u - win.refill_at(q);
        if constexpr (Ev::kLastDr) {
            run_ticks(ev, r, u, live_m, limit, [&]() {
                ++tick;
                tally.body(live_m);
                const uint64_t bail_m = wave_mask(r > u.bailout) & live_m;
                tally.bail(bail_m);
                // Lanes that have now run max_iters - 1 bodies without bailing:
                // their max_iters-th body is the dr update alone (max_iters >= 2
                // here; max_iters == 1 ends at the start).
                const uint64_t cap_m = wave_mask(t0 == tick + 1u - u.max_iters) & live_m & ~bail_m;
                tally.body(cap_m);
                const uint64_t done_m = cap_m | bail_m;
                last_m |= cap_m;
                if (sink.wants_k() && done_m != 0) {
                    if (__builtin_amdgcn_inverse_ballot_w64(done_m))
                        kh = tick - t0 + (__builtin_amdgcn_inverse_ballot_w64(cap_m) ? 1u : 0u);
                }
                live_m &= ~done_m;
                hold_m |= done_m;
            });
        } else {
            do {
                // Lanes making their max_iters-th body in this tick (max_iters >= 1).
                const uint64_t cap_m = wave_mask(t0 == tick + 1u - u.max_iters) & live_m;
                const float rn = tick_full(ev, r, u, live_m, cap_m);
                ++tick;
                tally.body(live_m);
                const uint64_t bail_m = wave_mask(rn > u.bailout) & live_m & ~cap_m;
                tally.bail(bail_m);
                const uint64_t done_m = cap_m | bail_m;
                if (sink.wants_k() && done_m != 0) {
                    if (__builtin_amdgcn_inverse_ballot_w64(done_m)) kh = tick - t0;
                }
                live_m &= ~done_m;
                hold_m |= done_m;
            } while ((uint32_t)__popcll(live_m) > limit);
        }
    }
    tally.flush(q.stats);
    if (q.dynamic) wave_retire(q);
}

}  // namespace cth
