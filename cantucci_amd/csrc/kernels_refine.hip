// Level-synchronous octree refinement on the GPU.
//
// The reference refines a CPU octree one leaf at a time (ShapeMesh::update,
// src/mesh/mod.rs:82-178, child spans from create_spans,
// src/octree/mod.rs:315-329).  Here the top of the tree, levels of up to
// top_nodes() nodes, is one workgroup's launch, and each level below it one
// batch: the centre distance of every node at depth d is evaluated by the
// lane-refill work loop, the split flags are prefix-summed, and every split
// node writes its 8 children (create_spans order) into the next level's array.
// Parents stay in level order, so the level-d array equals the oracle's
// breadth-first order.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <vector>

#include "internal.h"
#include "launch.h"
#include "point_sources.h"
#include "work_loop.h"

namespace cth {

// Node centre: start + (end - start) / 2 (SpanExt::center, src/octree/mod.rs:21-23);
// halving is exact, so `* 0.5f` equals the reference's `/ 2.0`.
struct SrcCenters {
    const float* spans;
    float power;
    __device__ __forceinline__ void get(uint32_t i, float& x, float& y, float& z, float& p) const {
        const float* sp = spans + 6 * (size_t)i;
        x = sp[0] + (sp[3] - sp[0]) * 0.5f;
        y = sp[1] + (sp[4] - sp[1]) * 0.5f;
        z = sp[2] + (sp[5] - sp[2]) * 0.5f;
        p = power;
    }
};

// Split rule of the refinement policy: |DE(centre)| < half diagonal, or NaN.
struct SinkSplit {
    uint32_t* flags;
    float half_diag;
    __device__ __forceinline__ static constexpr bool wants_k() { return false; }
    template <class E>
    __device__ __forceinline__ void put(uint32_t i, float d, uint32_t, float, float, const E&) const {
        flags[i] = ((d != d) || (fabsf(d) < half_diag)) ? 1u : 0u;
    }
};

__global__ void k_sphere_split(const float* nodes, uint32_t n, float cx, float cy, float cz, float radius,
                               float half_diag, uint32_t* flags) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    SrcCenters src{nodes, 0.0f};
    float x, y, z, p;
    src.get(i, x, y, z, p);
    const float c[3] = {cx, cy, cz};
    float d = sphere_de(x, y, z, c, radius);
    flags[i] = ((d != d) || (fabsf(d) < half_diag)) ? 1u : 0u;
}

__global__ void k_fill_u32(uint32_t* p, uint32_t n, uint32_t v) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Fill kernel for code that may be captured into a graph (a recorded memset
// node is avoided there).
int launch_fill_u32(uint32_t* p, size_t n, uint32_t v, hipStream_t st) {
    const size_t step = size_t(1) << 30;
    for (size_t off = 0; off < n; off += step) {
        uint32_t m = (uint32_t)((n - off) < step ? (n - off) : step);
        hipLaunchKernelGGL(k_fill_u32, dim3((m + 255) / 256), dim3(256), 0, st, p + off, m, v);
        int rc = check_hip(hipGetLastError(), "fill launch");
        if (rc) return rc;
    }
    return CTH_OK;
}

// One thread per (node, child): child c of a split node i lands at
// 8 * (incl[i] - 1) + c, incl being the inclusive prefix sum of the split
// flags.  create_spans (src/octree/mod.rs:315-329): centre
// = start + (end - start) / 2; child bit 2 = +x half, bit 1 = +y, bit 0 = +z.
__global__ void k_emit_children(const float* __restrict__ nodes, const uint32_t* __restrict__ flags,
                                const uint32_t* __restrict__ incl, uint32_t n, float* __restrict__ children) {
    uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t i = t >> 3, c = t & 7u;
    if (i >= n || !flags[i]) return;
    const float* sp = nodes + 6 * (size_t)i;
    float* out = children + 6 * ((size_t)(incl[i] - 1u) * 8 + c);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        float s = sp[a], e = sp[3 + a];
        float ctr = s + (e - s) * 0.5f;
        bool hi = (c >> (2 - a)) & 1u;
        out[a] = hi ? ctr : s;
        out[3 + a] = hi ? e : ctr;
    }
}

__global__ void k_emit_leaves(const float* __restrict__ nodes, const uint32_t* __restrict__ flags,
                              const uint32_t* __restrict__ incl, uint32_t n, float* __restrict__ leaves,
                              uint64_t cap) {
    uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t i = t / 6, a = t - i * 6;
    if (i >= n || !flags[i] || incl[i] - 1u >= cap) return;
    leaves[6 * (size_t)(incl[i] - 1u) + a] = nodes[6 * (size_t)i + a];
}

// The tree's top, all levels of at most top_nodes() (launch.h) nodes, in one
// workgroup: no read-back and no launch between levels.  A level took 20-30 us
// whatever its size (four or five launches and a wait for its split count).
// Depth 2, 4, 5 and 7 of the octree: 82, 129, 158, 226 -> 27, 55, 98, 167 us.
constexpr uint32_t kTopThreads = 1024;
constexpr uint32_t kMaxDepth = 20;
static_assert(2 + kMaxDepth + 1 <= kPinnedWords, "level counts fit");

struct RefineTop {
    float root[6];
    float half_diag[kMaxDepth + 1];
    uint32_t min_depth, max_depth;
    uint32_t top_nodes;
    float* nodes[2];   // level d in nodes[d & 1]
    float* leaves;     // nullable
    uint64_t cap;
    uint64_t* out;     // host memory: next depth (max_depth + 1: done), its nodes (or the leaves), nodes per level
};

template <class Ev>
__global__ __launch_bounds__(kTopThreads) void k_refine_top(RefineTop a, MandelUniform u) {
    __shared__ uint32_t wsum[kTopThreads / 64];
    const uint32_t wave = threadIdx.x >> 6;
    if (threadIdx.x < 6) a.nodes[0][threadIdx.x] = a.root[threadIdx.x];
    __syncthreads();
    uint32_t n = 1, depth = 0;
    for (;; ++depth) {
        const float* cur = a.nodes[depth & 1u];
        float* next = a.nodes[(depth & 1u) ^ 1u];
        const bool last = depth == a.max_depth;
        if (threadIdx.x == 0) a.out[2 + depth] = n;
        uint32_t total = 0;
        for (uint32_t base = 0; base < n; base += kTopThreads) {
            const uint32_t i = base + threadIdx.x;
            const bool valid = i < n;
            bool split = valid;
            if (depth >= a.min_depth) {
                // One evaluation per lane, as in the work loops (every lane
                // starts at once, so all reach the iteration cap together).
                Ev ev;
                float r = idle_start(ev, u);
                if (valid) {
                    float x, y, z, p;
                    SrcCenters{cur, u.power}.get(i, x, y, z, p);
                    ev.start(x, y, z, p, u);
                    r = ev.mag();
                }
                uint64_t live_m = wave_mask(valid && !(r > u.bailout));
                for (uint32_t k = 1; live_m != 0; ++k) {
                    const bool cap = k == u.max_iters;
                    const float rn = tick_full(ev, r, u, live_m, cap ? live_m : 0);
                    live_m = cap ? 0 : live_m & ~wave_mask(rn > u.bailout);
                }
                const float d = ev.finish(r);
                split = valid && ((d != d) || fabsf(d) < a.half_diag[depth]);
            }
            const uint64_t m = wave_mask(split);
            if ((threadIdx.x & 63u) == 0) wsum[wave] = (uint32_t)__popcll(m);
            __syncthreads();
            uint32_t rank = total + lane_rank(m);
            for (uint32_t w = 0; w < kTopThreads / 64; ++w) {
                rank += w < wave ? wsum[w] : 0u;
                total += wsum[w];
            }
            if (split && last) {
                if (a.leaves && rank < a.cap) {
#pragma unroll
                    for (int k = 0; k < 6; ++k) a.leaves[6 * (size_t)rank + k] = cur[6 * i + k];
                }
            } else if (split) {
                float sp[6], ctr[3];
#pragma unroll
                for (int k = 0; k < 6; ++k) sp[k] = cur[6 * i + k];
#pragma unroll
                for (int k = 0; k < 3; ++k) ctr[k] = sp[k] + (sp[3 + k] - sp[k]) * 0.5f;
                float* out = next + 48 * (size_t)rank;
#pragma unroll
                for (uint32_t c = 0; c < 8; ++c) {
#pragma unroll
                    for (int k = 0; k < 3; ++k) {
                        const bool hi = (c >> (2 - k)) & 1u;
                        out[6 * c + k] = hi ? ctr[k] : sp[k];
                        out[6 * c + 3 + k] = hi ? sp[3 + k] : ctr[k];
                    }
                }
            }
            __syncthreads();  // wsum is rewritten; after the last round, the level's children are complete
        }
        if (last) {
            if (threadIdx.x == 0) {
                a.out[0] = depth + 1;
                a.out[1] = total;
            }
            return;
        }
        n = 8 * total;
        if (n == 0 || n > a.top_nodes) break;
    }
    if (threadIdx.x == 0) {
        a.out[0] = depth + 1;
        a.out[1] = n;
    }
}

static inline uint32_t cdiv32(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }

// Level-synchronous refinement: the top of the tree in one launch, then per
// level the split flags (forced, sphere closed form or a DE refill launch), an
// inclusive scan of the flags, one 4-byte read-back of the split count into
// pinned host memory, and the children.  Node, flag, offset and scan buffers are
// the context's scratch slots (ping-pong for the nodes), so a level allocates
// nothing.
int refine_levels(Ctx& c, const cth_shape& s, const float* root, uint32_t min_depth, uint32_t max_depth,
                  const float* half_diag, float* leaves, size_t cap, size_t* nleaves, uint64_t* level_counts,
                  hipStream_t st) {
    MandelUniform u{};
    int family = FAM_SPHERE;
    if (s.kind != CTH_SHAPE_SPHERE) {
        int rc = resolve_mandel(s, u, family);
        if (rc) return rc;
    }
    const uint64_t kMaxNodes = 1ull << 28;
    *nleaves = 0;
    uint32_t depth = 0;
    uint64_t n = 1;
    float* nodes[2] = {};
    const bool top_launch = !c.stats;  // counted work goes through the work loops
    const size_t first = top_launch ? (size_t)8 * kTopNodes : 1;
    int rc = CTH_OK;
    for (int k = 0; k < 2 && !rc; ++k) rc = c.scratch(WS_NODES_A + k, first * 6 * sizeof(float), (void**)&nodes[k]);
    if (rc) return fail(rc, "refinement scratch allocation failed");
    if (top_launch) {
        RefineTop top{};
        std::copy(root, root + 6, top.root);
        std::copy(half_diag, half_diag + max_depth + 1, top.half_diag);
        top.min_depth = min_depth;
        top.max_depth = max_depth;
        top.top_nodes = top_nodes(family == FAM_SPHERE ? 1u : u.max_iters, family == FAM_TRIG && !u.integral);
        top.nodes[0] = nodes[0];
        top.nodes[1] = nodes[1];
        top.leaves = leaves;
        top.cap = cap;
        top.out = c.pinned;
        if (family == FAM_SPHERE) {
            u.max_iters = 1;
            u.bailout = 0.0f;
            for (int a = 0; a < 3; ++a) u.center[a] = s.center[a];
            u.radius = s.radius;
            hipLaunchKernelGGL(k_refine_top<SphereEv>, dim3(1), dim3(kTopThreads), 0, st, top, u);
        } else if (family == FAM_P8) {
            with_p8(c.mode, [&](auto ev) {
                hipLaunchKernelGGL(k_refine_top<decltype(ev)>, dim3(1), dim3(kTopThreads), 0, st, top, u);
            });
        } else {
            hipLaunchKernelGGL(k_refine_top<TrigExact>, dim3(1), dim3(kTopThreads), 0, st, top, u);
        }
        rc = check_hip(hipGetLastError(), "refinement top launch");
        int rs = check_hip(hipStreamSynchronize(st), "sync");
        if (rc || rs) return rc ? rc : rs;
        depth = (uint32_t)c.pinned[0];
        n = c.pinned[1];
        for (uint32_t d = 0; d < depth && level_counts; ++d) level_counts[d] = c.pinned[2 + d];
        if (depth > max_depth) {
            *nleaves = n;
            return CTH_OK;
        }
    } else {
        rc = check_hip(hipMemcpyAsync(nodes[0], root, 6 * sizeof(float), hipMemcpyHostToDevice, st), "H2D root");
    }
    int slot = WS_NODES_A + (int)(depth & 1u);
    float* cur = nodes[depth & 1u];
    for (; depth <= max_depth && rc == CTH_OK; ++depth) {
        if (level_counts) level_counts[depth] = n;
        if (n == 0) {
            for (uint32_t d2 = depth + 1; d2 <= max_depth && level_counts; ++d2) level_counts[d2] = 0;
            break;
        }
        uint32_t* flags = nullptr;
        uint32_t* incl = nullptr;
        if (c.scratch(WS_FLAGS, n * sizeof(uint32_t), (void**)&flags) ||
            c.scratch(WS_OFFS, n * sizeof(uint32_t), (void**)&incl)) {
            rc = fail(CTH_E_NOMEM, "refinement scratch allocation failed");
            break;
        }
        if (depth < min_depth) {
            hipLaunchKernelGGL(k_fill_u32, dim3(cdiv32(n, 256)), dim3(256), 0, st, flags, (uint32_t)n, 1u);
            rc = check_hip(hipGetLastError(), "fill launch");
        } else if (family == FAM_SPHERE) {
            hipLaunchKernelGGL(k_sphere_split, dim3(cdiv32(n, 256)), dim3(256), 0, st, cur, (uint32_t)n, s.center[0],
                               s.center[1], s.center[2], s.radius, half_diag[depth], flags);
            rc = check_hip(hipGetLastError(), "sphere split launch");
        } else {
            SrcCenters src{cur, s.power};
            SinkSplit sink{flags, half_diag[depth]};
            rc = run_refill(c, family, u, src, sink, (uint32_t)n, st, level_shape(c.shape_spans));
        }
        if (rc) break;
        size_t temp_bytes = 0;
        rc = check_hip(hipcub::DeviceScan::InclusiveSum(nullptr, temp_bytes, flags, incl, (int)n, st), "scan size");
        void* temp = nullptr;
        if (!rc && c.scratch(WS_SCAN, temp_bytes, &temp)) rc = fail(CTH_E_NOMEM, "scan scratch allocation failed");
        if (!rc) rc = check_hip(hipcub::DeviceScan::InclusiveSum(temp, temp_bytes, flags, incl, (int)n, st), "scan");
        if (!rc)
            rc = check_hip(hipMemcpyAsync(c.pinned, incl + (n - 1), sizeof(uint32_t), hipMemcpyDeviceToHost, st),
                           "D2H split count");
        if (!rc) rc = check_hip(hipStreamSynchronize(st), "sync");
        if (rc) break;
        const uint64_t split = *reinterpret_cast<volatile uint32_t*>(c.pinned);
        if (depth == max_depth) {
            *nleaves = split;
            if (leaves && split) {
                hipLaunchKernelGGL(k_emit_leaves, dim3(cdiv32(n * 6, 256)), dim3(256), 0, st, cur, flags, incl,
                                   (uint32_t)n, leaves, (uint64_t)cap);
                rc = check_hip(hipGetLastError(), "leaves launch");
            }
            break;
        }
        const uint64_t next_n = split * 8;
        if (next_n > kMaxNodes) {
            rc = fail(CTH_E_INVALID, "refinement exceeds 2^28 nodes in one level");
            break;
        }
        // The next level goes to the other node slot; growing that slot
        // waits for the device, so `cur` stays valid.
        const int next_slot = (slot == WS_NODES_A) ? WS_NODES_B : WS_NODES_A;
        float* next = nullptr;
        if (c.scratch(next_slot, next_n * 6 * sizeof(float) + 4, (void**)&next)) {
            rc = fail(CTH_E_NOMEM, "refinement scratch allocation failed");
            break;
        }
        if (next_n) {
            hipLaunchKernelGGL(k_emit_children, dim3(cdiv32(n * 8, 256)), dim3(256), 0, st, cur, flags, incl,
                               (uint32_t)n, next);
            rc = check_hip(hipGetLastError(), "children launch");
        }
        cur = next;
        slot = next_slot;
        n = next_n;
    }
    int rs = check_hip(hipStreamSynchronize(st), "sync");
    return rc ? rc : rs;
}

}  // namespace cth
