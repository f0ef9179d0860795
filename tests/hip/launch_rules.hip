// The host rules of a launch (make_queue and the counter entries it takes),
// checked on the CPU: no kernel is compiled or launched, and the capture state
// of a stream is the test's own.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <vector>

static bool g_capturing = false;
static hipError_t test_stream_is_capturing(hipStream_t, hipStreamCaptureStatus* s) {
    *s = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
#define hipStreamIsCapturing test_stream_is_capturing
#include "launch.h"
#include "tangent.h"

namespace cth {
CapturePool& capture_pool() {
    static CapturePool p;
    return p;
}
}  // namespace cth
using namespace cth;

static int g_failed = 0;
#define CHECK(x)                                                                                       \
    do {                                                                                               \
        if (!(x)) {                                                                                    \
            std::printf("%s:%d: %s\n", __FILE__, __LINE__, #x);                                        \
            ++g_failed;                                                                                \
        }                                                                                              \
    } while (0)

static Ctx make_ctx(std::vector<uint32_t>& ring) {
    ring.assign(counter_words(COUNTER_RING), 0);
    Ctx c;
    c.num_cus = 256;
    c.counters = ring.data();
    return c;
}
static const hipStream_t kStream = (hipStream_t)0x1000, kOther = (hipStream_t)0x2000;

static WorkQueue queue(Ctx& c, uint32_t total, const LaunchShape& ls, hipStream_t st,
                       WaveSpread spread = P8Exact::kSpread) {
    uint32_t blocks = 0;
    return make_queue(c, total, ls, spread, blocks, st);
}

// A launch into a graph that owns no counters takes no entry of the ring and
// claims nothing: default static shapes, default claiming ones and shapes set
// by the caller.  One recorded through the pool takes the graph's own entries.
static void captures() {
    std::vector<uint32_t> ring, own(counter_words(GRAPH_ENTRIES), 0);
    Ctx c = make_ctx(ring);
    const LaunchShape given{256, 8, 256, 32, 1, true};
    const LaunchShape shapes[] = {c.shape_de,  c.shape_spans, c.shape_trace, c.shape_adj,
                                  c.shape_jobs, c.shape_mesh, given};
    for (const LaunchShape& ls : shapes) {
        for (uint32_t total : {1u, 100000u, 20000000u}) {
            for (hipStream_t st : {kStream, (hipStream_t) nullptr}) {
                g_capturing = false;
                const WorkQueue eager = queue(c, total, ls, st);
                CHECK(eager.dynamic == (eager.ctr != nullptr));
                if (total == 20000000u) CHECK(eager.dynamic);
                if (total == 1u) CHECK(!eager.dynamic);
            }
            g_capturing = true;
            const uint32_t pos = c.ring_pos;
            const WorkQueue q = queue(c, total, ls, kStream);
            CHECK(!q.dynamic && !q.ctr && c.ring_pos == pos);
            CHECK((uint64_t)q.chunk * q.chunks >= total && (uint64_t)q.chunk * (q.chunks - 1) < total);
            capture_pool().stream = kStream;
            capture_pool().counters = own.data();
            const WorkQueue g = queue(c, total, ls, kStream), f = queue(c, total, ls, kOther);
            CHECK(!g.dynamic || (g.ctr >= own.data() && g.ctr < own.data() + own.size()));
            if (total == 20000000u) CHECK(g.dynamic);
            CHECK(!f.dynamic && c.ring_pos == pos);  // a stream forked off the captured one
            capture_pool() = CapturePool{};
            g_capturing = false;
        }
    }
}

// A launch takes an entry of the ring only if it has more chunks than waves: of
// 8^3-cell spans on one wave per CU, 30 take one, one takes none.  The ring comes
// round after COUNTER_RING entries.
static void ring_advances() {
    std::vector<uint32_t> ring;
    Ctx c = make_ctx(ring);
    const LaunchShape thin{64, 1, 64, 32, 1, true}, full{256, 8, 256, 32, 1, true};
    const WorkQueue first = queue(c, 3000 * 729, full, kStream);
    CHECK(first.dynamic && c.ring_pos == 1);
    for (uint32_t i = 1; i < COUNTER_RING; ++i) {
        CHECK(!queue(c, 729, thin, kStream).ctr);
        const WorkQueue q = queue(c, 30 * 729, thin, kStream);
        CHECK(q.dynamic && q.ctr != first.ctr && c.ring_pos == i + 1);
    }
    CHECK(queue(c, 3000 * 729, full, kOther).ctr == first.ctr);
}

// The reverse sweep's two kernels run on single-wave workgroups, at most eight to
// a CU and no more than the shape allows, whatever the size.
static void orbit_sweep() {
    std::vector<uint32_t> ring;
    Ctx c = make_ctx(ring);
    for (uint32_t n : {1u, 64u, 65u, 5000u, 262144u, 1048576u, 4194304u, 100000000u}) {
        uint32_t blocks = 0;
        const LaunchShape ls = single_waves(c.shape_adj);
        WorkQueue q = make_queue(c, n, ls, kOrbitSpread, blocks, kStream);
        CHECK(ls.block == 64 && blocks == q.waves && q.waves <= 8u * 256u);
        CHECK(q.waves == std::min((n + 63u) / 64u, 8u * 256u));
        q = make_queue(c, n, single_waves(LaunchShape{256, 1, 256, 32, 0, true}), kOrbitSpread, blocks, kStream);
        CHECK(blocks == q.waves && q.waves <= 4u * 256u);
    }
}

// The reverse sweep's one kernel claims from four chunks of 64 a wave on, and not
// at all where the caller's shape is static.
static void sweep_shapes() {
    for (uint32_t n : {1u, 300000u, 524287u, 524288u, 30000000u}) {
        CHECK(sweep_shape(LaunchShape{}, n, 256, 8).dynamic == (n >= 524288u));
        for (uint32_t dyn : {0u, 1u}) {
            const LaunchShape w = sweep_shape(LaunchShape{128, 16, 128, 32, dyn, true}, n, 256, 8);
            CHECK(w.given && w.dynamic == (dyn && n >= 524288u));
            CHECK(w.block == 64 && w.blocks_per_cu == 32 && w.chunk == 128);
        }
    }
}

// A tangent launch of at most a wave per CU gives every wave a workgroup of its
// own, unless the caller has set the shape.
static void tangent_shapes() {
    std::vector<uint32_t> ring;
    Ctx c = make_ctx(ring);
    for (uint32_t n : {1u, 64u, 65u, 5000u, 16384u, 16385u, 4000000u}) {
        uint32_t blocks = 0;
        const LaunchShape ls = tangent_shape(c.shape_adj, n, 256);
        const WorkQueue q = make_queue(c, n, ls, P8Tangent::kSpread, blocks, kStream);
        CHECK(ls.block == (n <= 16384u ? 64 : c.shape_adj.block));
        CHECK(q.waves == blocks * (ls.block / 64u) && (n > 16384u || blocks == (n + 63u) / 64u));
        const LaunchShape set{256, 4, 128, 16, 0, true};
        CHECK(tangent_shape(set, n, 256).block == 256);
    }
}

// The refinement's one workgroup takes the whole levels it has room for, fewer
// nodes the longer their evaluations are.
static void refinement_tops() {
    for (bool real : {false, true}) {
        uint32_t was = kTopNodes;
        for (uint32_t it : {1u, 15u, 28u, 29u, 64u, 65u, 512u, 513u, 4000u}) {
            const uint32_t n = top_nodes(it, real);
            CHECK(n <= was && n >= 64 && n <= kTopNodes);
            was = n;
        }
    }
    CHECK(top_nodes(15, true) == 2048 && top_nodes(129, false) == 512 && top_nodes(129, true) == 64);
}

// One kernel while it is the faster one: at every size up to `any` iterations,
// with fewer points beyond.
static void sweep_kernels() {
    for (uint32_t any : {16u, 20u, 22u}) {
        for (uint32_t n : {1u, 1u << 17, 1u << 18, 1u << 20, 1u << 22}) {
            for (uint32_t it = 1; it <= any; ++it) CHECK(one_sweep_kernel(it, n, any));
            for (uint32_t it = any + 1; it <= 40; ++it) {
                const bool one = one_sweep_kernel(it, n, any);
                CHECK(one == (n <= 1u << 17 ? it <= 32 : n <= 1u << 18 && it <= 21));
            }
        }
        CHECK(!one_sweep_kernel(32, (1u << 17) + 1, any) && !one_sweep_kernel(24, 1000000, any));
        CHECK(!one_sweep_kernel(4095, 1, any));
    }
}

static bool same(const WorkQueue& a, const WorkQueue& b) {
    return a.waves == b.waves && a.chunk == b.chunk && a.chunks == b.chunks && a.rotate == b.rotate &&
           a.dynamic == b.dynamic && a.refill_min == b.refill_min;
}

// A shape that was read and is set back, also after another, leaves every launch
// as it was; the caller's static and claiming shapes are kept in all sizes.
static void shapes_kept() {
    std::vector<uint32_t> r0, r1;
    Ctx c = make_ctx(r0), d = make_ctx(r1);
    for (int k : {CTH_KERNEL_DE, CTH_KERNEL_TRACE, CTH_KERNEL_ADJOINT, CTH_KERNEL_SPANS, CTH_KERNEL_JOBS,
                  CTH_KERNEL_MESH}) {
        LaunchShape *a = c.launch_shape(k), *b = d.launch_shape(k);
        const cth_launch was = b->get();
        b->set({128, 3, 128, 7, 1});
        b->set(was);
        for (uint32_t n : {1u, 300000u, 4000000u, 30000000u}) {
            CHECK(same(queue(c, n, *a, kStream), queue(d, n, *b, kStream)));
            for (int dyn : {0, 1}) {
                LaunchShape s;
                s.set({256, 16, 256, 32, (uint32_t)dyn});
                CHECK(s.get().dynamic == (uint32_t)dyn);
                const WorkQueue q = queue(c, n, s, kStream);
                CHECK(!q.dynamic || dyn);
                CHECK(q.chunk <= 256u);
                CHECK(n != 30000000u || q.dynamic == (uint32_t)dyn);
            }
        }
    }
}

// A refinement level is launched the same on a default span shape and on one
// set by the caller: static, and claiming from 4 chunks of 128 a wave on.
static void refinement_levels() {
    std::vector<uint32_t> ring;
    Ctx c = make_ctx(ring);
    LaunchShape set = c.shape_spans;
    set.given = true;
    for (uint32_t n : {1u, 100000u, 4194303u, 4194304u, 200000000u}) {
        const WorkQueue q = queue(c, n, level_shape(c.shape_spans), kStream);
        CHECK(same(q, queue(c, n, level_shape(set), kStream)));
        CHECK(q.dynamic == (n >= 4194304u));
        CHECK(q.dynamic || q.chunk == 64u);
    }
}

// Lanes without a point in a launch with a power per point run the shortest
// power ladder (powi_ladder halves its exponent once per turn), not powf.
static void idle_power() {
    const int n = (int)kPointPower;
    CHECK((float)n == kPointPower && n >= 1 && n < 64);
    CHECK(n / 2 == 0);
}

int main() {
    idle_power();
    refinement_levels();
    captures();
    shapes_kept();
    tangent_shapes();
    refinement_tops();
    sweep_kernels();
    sweep_shapes();
    orbit_sweep();
    ring_advances();
    std::printf(g_failed ? "%d checks failed\n" : "launch rules ok\n", g_failed);
    return g_failed ? 1 : 0;
}
