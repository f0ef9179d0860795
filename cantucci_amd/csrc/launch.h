// Launch plumbing shared by the kernel units: the lane-refill kernel
// template and the persistent-grid sizing.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>

#include "internal.h"
#include "point_sources.h"
#include "work_loop.h"

namespace cth {

// Ev::kWavesPerSimd: the occupancy the evaluator's register budget is fitted
// to (the P8 evaluators fit 64 VGPRs, 8 waves per SIMD, without spilling).
// kCount: the counting instantiation (work tallies, see WorkTally).
template <class Ev, class Src, class Sink, bool kCount = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(Ev::kWavesPerSimd))) void k_refill(
    Src src, MandelUniform u, Sink sink, WorkQueue q) {
    refill_loop<Ev, kCount>(src, u, sink, q);
}

// Sphere: no iteration, one point per thread.
template <class Src>
__global__ __launch_bounds__(256) void k_sphere(Src src, uint32_t n, float cx, float cy, float cz, float radius,
                                                float* out, uint32_t* iters) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float x, y, z, p;
    src.get(i, x, y, z, p);
    const float c[3] = {cx, cy, cz};
    out[i] = sphere_de(x, y, z, c, radius);
    if (iters) iters[i] = 0;
}

// Whether `st` is being captured into a graph that owns no counter entries.  Its
// replays would claim from the entry of the context's ring that the capture took,
// beside the launches in flight that the ring has come round to, and from freed
// memory once the context is gone: no launch claims there, whatever its shape.
inline bool foreign_capture(hipStream_t st) { return capture_pool().stream != st && is_capturing(st); }

// A launch's workgroups and chunks.  Up to a chunk of `least` indices (64 or
// fewer) for each of spread.fill waves per CU a launch is spread as thinly as
// possible; from four chunks per wave on it grows to the launch shape's (and
// spread.most) waves.  In between it stays at `fill` up to 8/3 chunks a wave: a lane that takes a
// second point while its wave's slowest is still iterating costs little, more
// waves on a SIMD cost their share of its issue slots.  Then evaluators with
// spread.grow grow to that: 500,000 / 600,000 / 800,000 tangent normals at power
// 5 59 / 73 / 87 -> 46 / 56 / 67 us (growing from four chunks on), 0.8 / 1 / 1.2 M
// points 34.8 / 44.0 / 51.0 -> 31.5 / 36.2 / 44.8; 20 or 24 waves per CU from the
// start cost 300,000 points 9 %.
//
// Measured on the default shapes, us per launch (in parentheses with the
// workgroup count taken from the configured 256-index chunk): 64^3 grid 10.5
// (24.6), 2 M points at power 8 34.5 (47), 700,000 at power 5 33 (49; 47 at
// fill 32), tangent normals of 300,000 points with powers 48 (68; 69 at fill
// 16), of 2 M points 153 (195; 175 without `most`).
//
// A default static shape lets its waves claim once each of the waves that fit
// on the chip (8 per SIMD, or spread.most) has 4 chunks of 128: 8 workgroups per
// CU, chunks of up to 1024, which evens out regions that a static deal gives to
// a few waves.  Below, the claims and their smaller share of first chunks cost
// more than that gives.  Static / claimed, us: 256^3 grid 177 / 147, 164^3 (just
// over the line) 64.7 / 54.1, 112^3 24.4 / 26.1; 4 M points at power 5
// 164 / 147, of tangent normals 252 / 228, 2^18 44 / 46; 4 poses of 1080p
// 1987 / 1550, one 848 / 844; 24 mixed jobs 1796 / 1400.  Chunks of 64 take
// twice the claims (200^3 grid at 6 iterations 76 us, static 73, with 128 66).
inline WorkQueue make_queue(Ctx& c, uint32_t total, LaunchShape ls, WaveSpread spread, uint32_t& blocks,
                            hipStream_t st, uint32_t least = 64) {
    constexpr uint32_t kLeastClaim = 128;
    const uint64_t resident = (uint64_t)c.num_cus * std::min(32u, spread.most);
    uint64_t lowest = 64;
    const bool large = !ls.given && !ls.dynamic && total >= 4u * kLeastClaim * resident;
    const bool claims = (ls.dynamic || large) && !foreign_capture(st);
    if (large && claims) {
        ls.blocks_per_cu = 8 * (256 / ls.block);
        ls.chunk = 1024;
        lowest = kLeastClaim;
    }
    const uint64_t cus = (uint64_t)c.num_cus, waves_per_block = (uint64_t)ls.block / 64u;
    const uint64_t small = ((uint64_t)total + least - 1) / least;
    // Whole workgroups for each CU (16.02 waves per CU cost 700,000 points at
    // power 5 4 %), the nearest to 3/8 wave for each chunk.
    const uint64_t per_cu = (small * 3u / 8u + cus * waves_per_block / 2u) / (cus * waves_per_block) * waves_per_block;
    uint64_t waves = std::max({std::min(small, cus * spread.fill), cus * std::min<uint64_t>(per_cu, spread.grow),
                               std::min(small / 4u, cus * spread.most)});
    blocks = (uint32_t)std::max<uint64_t>(
        1, std::min(cus * (uint64_t)ls.blocks_per_cu, (waves + waves_per_block - 1) / waves_per_block));
    WorkQueue q;
    q.waves = blocks * (uint32_t)waves_per_block;
    q.total = total;
    // About 8 chunks per wave, so that launches still balance:
    // chunk = clamp(total / (8 waves), lowest, configured), a multiple of 64.
    uint64_t fair = (uint64_t)total / ((uint64_t)q.waves * 8u);
    uint64_t ch = std::min<uint64_t>(ls.chunk, std::max(lowest, fair));
    q.chunk = least < 64 ? least : (uint32_t)(ch & ~63ull);
    q.chunks = (uint32_t)(((uint64_t)total + q.chunk - 1) / q.chunk);
    q.refill_min = ls.refill_min < 1 ? 1 : (ls.refill_min > 64 ? 64 : ls.refill_min);
    // Only chunks beyond every wave's first are claimed.
    q.dynamic = claims && q.chunks > q.waves ? 1u : 0u;
    // Static rows rotate from four rows on (128^3 grid 47 -> 42 us, 24 mixed
    // jobs 2.27 -> 1.85 ms).  With fewer, the waves of the partial last row
    // decide, and the first waves, which start first, are the best ones for it
    // (96^3 grid 17 us, rotated 22).
    q.rotate = q.chunks >= 4ull * q.waves ? (uint32_t)(q.waves * 0.381966f) : 0u;
    q.shards = 1;
    while (q.shards < kMaxShards && 2 * q.shards <= blocks) q.shards *= 2;
    q.ctr = q.dynamic ? c.take_counters(st) : nullptr;
    q.stats = c.stats;
    return q;
}

// The largest level that the refinement's one workgroup takes (k_refine_top).
// Beyond, a level's own launches are faster: one CU's waves share its issue
// slots, and long evaluations take longer there than the launches cost (64 nodes
// are a single wave, which takes as long anywhere).  Depths 2 to 4 of the octree
// at 64 / 512 / 2,048 nodes, us: power 8 at 15, 60, 129, 300, 1000
// iterations 162 / 127 / 109, 240 / 207 / 250, 355 / 330 / 469, 648 / 635 / 1009,
// 1838 / 1883 / 3220; power 5 183 / 150 / 151, 306 / 279 / 278, 490 / 476 / 476,
// 946 / 963 / 962, 2813 / 2952 / 2951; a real power 245 / 220 / 220, 567 / 570 /
// 570, 1061 / 1106 / 1106, 2280 / 2433 / 2432, 7292 / 7866 / 7870.
constexpr uint32_t kTopNodes = 2048;
inline uint32_t top_nodes(uint32_t max_iters, bool real_power) {
    if (max_iters <= 28) return kTopNodes;
    return max_iters <= (real_power ? 64u : 512u) ? 512u : 64u;
}

// A refinement level's launch: the span family's shape with 64-point chunks dealt
// statically, which spreads a level over the whole chip; levels of millions of
// nodes claim as every default shape does, whether the span shape is the caller's
// or not (depth 10 of the octree, 16 M nodes: static 2.78 ms, so 2.50).
inline LaunchShape level_shape(LaunchShape spans) {
    spans.chunk = 64;
    spans.dynamic = 0;
    spans.given = false;
    return spans;
}

// Whether the reverse sweep of n points runs in one kernel (orbits in LDS) or in
// two (orbits in memory).  The LDS leaves fewer waves per CU with every
// iteration, which costs nothing while there are few points for each CU; `any`
// is the cap up to which one kernel is the better one at every size: 22 at
// power 8, 20 at another integer power of the launch, 16 with real powers, whose
// steps are the longest and want the most waves.  A call on points spread evenly
// over the cube, us, two kernels (the workspace's allocation included) / one:
//   iterations    18         20         22         24         28         32
//   P8   2^17     57 / 30    54 / 32    58 / 38    60 / 41    59 / 47    85 / 53
//        2^18     72 / 37    75 / 40    77 / 63    80 / 66    86 / 100   91 / 112
//        2^20    152 / 136  162 / 140  166 / 165  172 / 193  192 / 236  201 / 257
//        2^22    641 / 425  632 / 476  657 / 555  679 / 660  729 / 828  791 / 898
//   p5   2^18     82 / 49    86 / 52    89 / 85    94 / 94   101 / 124  108 / 139
//        2^20    174 / 184  187 / 188  194 / 219  200 / 260  227 / 319  232 / 349
//        2^22    657 / 594  665 / 657  703 / 768  714 / 909  811 / 1142 860 / 1238
//   real 2^17     72 / 51    76 / 57    87 / 66    89 / 72    98 / 82   127 / 93
//        2^18     99 / 64   104 / 69   109 / 115  115 / 123  125 / 165  136 / 185
//        2^20    209 / 237  223 / 249  235 / 288  245 / 343  275 / 427  300 / 474
//        2^22    740 / 781  773 / 868  820 / 1025 880 / 1218 955 / 1540 1056 / 1694
// (15 iterations, 2^20: 136 / 118, 155 / 154, 185 / 196; 2^22: 584 / 364,
// 590 / 494, 658 / 644.)
inline bool one_sweep_kernel(uint32_t max_iters, uint32_t n, uint32_t any) {
    return max_iters <= (n <= 1u << 17 ? 32u : n <= 1u << 18 ? std::max(any, 21u) : any);
}

// The family's shape in workgroups of a single wave, with as many waves per CU
// (the reverse sweep's, and small tangent launches').
inline LaunchShape single_waves(LaunchShape ls) {
    ls.blocks_per_cu *= ls.block / 64;
    ls.block = 64;
    return ls;
}

// Its one kernel (orbits in LDS), for n points on at least `fill` waves per CU:
// what fits beside the orbits need not spread evenly over a CU's four SIMDs, so
// waves claim their chunks where there are enough to even that out (4 M points
// at 15 iterations 558 -> 469 us, 300,000 points 65 -> 73), unless the caller's
// shape is static.
inline LaunchShape sweep_shape(const LaunchShape& family, uint32_t n, int num_cus, uint32_t fill) {
    LaunchShape ls = single_waves(family);
    ls.dynamic = (!family.given || family.dynamic) && n / 256u >= (uint32_t)num_cus * fill;
    ls.given = true;
    return ls;
}

// Its two kernels (orbits in memory): a lane writes and reads its own orbit, 64
// rows to a wave, and the waves of a CU share its vector cache, so few waves are
// best and they start on CUs of their own.  Both kernels at 120 iterations, us,
// on four-wave workgroups with the forward kernels' spread -> so: power 8
// 5,000 points 233 -> 134, 2^18 298 -> 187, 2^20 1059 -> 431, 2^22 4077 -> 1770;
// per-point powers 396 -> 282, 597 -> 371, 1228 -> 803, 4737 -> 3212.  (The
// workspace's place in memory moves single figures by up to a quarter.)
constexpr WaveSpread kOrbitSpread{8, 8};

// A tangent evaluator's launch: on the default shape in single-wave workgroups
// while there is at most one wave for each CU, since the four waves of a
// workgroup slow each other down on one CU (a body is 8 KB of code).  256 / 5,000 /
// 16,384 points, normals at power 5 and gradients with a power per point, 15
// iterations 21 / 30 / 22 and 29 / 40 / 31 -> 19 / 19 / 18 and 28 / 27 / 27 us, 60
// iterations 83 / 109 / 72 and 117 / 144 / 109 -> 68 / 62 / 62 and 102 / 96 / 96;
// power 8 within 1 us.
inline LaunchShape tangent_shape(const LaunchShape& family, uint64_t n, int num_cus) {
    return !family.given && n <= 64u * (uint64_t)num_cus ? single_waves(family) : family;
}

template <class Src, class Sink>
inline int run_refill(Ctx& c, int family, const MandelUniform& u, const Src& src, const Sink& sink,
                      uint32_t total, hipStream_t st, const LaunchShape& ls) {
    uint32_t blocks = 0;
    WorkQueue q = make_queue(c, total, ls, family == FAM_P8 ? P8Exact::kSpread : TrigExact::kSpread, blocks, st);
    dim3 grid(blocks), block(ls.block);
    if (family == FAM_P8) {
        with_p8(c.mode, [&](auto ev) {
            using Ev = decltype(ev);
            if (q.stats)
                hipLaunchKernelGGL((k_refill<Ev, Src, Sink, true>), grid, block, 0, st, src, u, sink, q);
            else
                hipLaunchKernelGGL((k_refill<Ev, Src, Sink>), grid, block, 0, st, src, u, sink, q);
        });
    } else if (q.stats) {
        hipLaunchKernelGGL((k_refill<TrigExact, Src, Sink, true>), grid, block, 0, st, src, u, sink, q);
    } else {
        hipLaunchKernelGGL((k_refill<TrigExact, Src, Sink>), grid, block, 0, st, src, u, sink, q);
    }
    return check_hip(hipGetLastError(), "refill kernel launch");
}

// Distances, with the loop-body counts where they are asked for.
template <class Src>
inline int run_dist(Ctx& c, int family, const MandelUniform& u, const Src& src, float* out, uint32_t* iters,
                    uint32_t total, hipStream_t st, const LaunchShape& ls) {
    return iters ? run_refill(c, family, u, src, SinkDistIters{out, iters}, total, st, ls)
                 : run_refill(c, family, u, src, SinkDist{out}, total, st, ls);
}

}  // namespace cth
