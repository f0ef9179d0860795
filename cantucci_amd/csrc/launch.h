// Launch plumbing shared by the kernel units: the lane-refill kernel
// template and the persistent-grid sizing.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>

#include "internal.h"
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

// Waves per CU that a small launch is spread over (8 per SIMD, what the P8
// kernels can hold).  At the configured chunk alone a 64^3 grid was 256
// workgroups, one wave per SIMD, and took 25 us; filled, 10 us.  One leaf's
// 65^3 corners: 60 -> 11 us; its 9,868 vertices' taps: 249 -> 26 us.
constexpr uint64_t kFillWaves = 32;

inline WorkQueue make_queue(Ctx& c, uint32_t total, const LaunchShape& ls, uint32_t& blocks, hipStream_t st) {
    // Workgroups: enough for the configured chunks, and for a small launch
    // enough that its 64-index chunks fill kFillWaves waves per CU.
    const uint64_t waves_per_block = (uint64_t)ls.block / 64u;
    const uint64_t per_block = 64u * waves_per_block;
    const uint64_t want = (uint64_t)c.num_cus * (uint64_t)ls.blocks_per_cu;
    const uint64_t full = ((uint64_t)total + ls.chunk * waves_per_block - 1) / (ls.chunk * waves_per_block);
    const uint64_t fill = std::min(((uint64_t)total + per_block - 1) / per_block,
                                   (uint64_t)c.num_cus * kFillWaves / waves_per_block);
    blocks = (uint32_t)std::max<uint64_t>(1, std::min(want, std::max(full, fill)));
    WorkQueue q;
    q.waves = blocks * (uint32_t)waves_per_block;
    q.total = total;
    // At least ~8 chunks per wave, so that small launches still balance:
    // chunk = clamp(total / (8 waves), 64, configured), a multiple of 64.
    uint64_t fair = (uint64_t)total / ((uint64_t)q.waves * 8u);
    uint64_t ch = std::min<uint64_t>(ls.chunk, std::max<uint64_t>(64, fair));
    q.chunk = (uint32_t)(ch & ~63ull);
    q.chunks = (uint32_t)(((uint64_t)total + q.chunk - 1) / q.chunk);
    q.refill_min = ls.refill_min < 1 ? 1 : (ls.refill_min > 64 ? 64 : ls.refill_min);
    // Only chunks beyond every wave's first are claimed.
    q.dynamic = ls.dynamic && q.chunks > q.waves ? 1u : 0u;
    q.shards = 1;
    while (q.shards < kMaxShards && 2 * q.shards <= blocks) q.shards *= 2;
    q.ctr = q.dynamic ? c.take_counters(st) : nullptr;
    q.stats = c.stats;
    return q;
}

template <class Src, class Sink>
inline int run_refill(Ctx& c, int family, const MandelUniform& u, const Src& src, const Sink& sink,
                      uint32_t total, hipStream_t st, const LaunchShape& ls) {
    uint32_t blocks = 0;
    WorkQueue q = make_queue(c, total, ls, blocks, st);
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

}  // namespace cth
