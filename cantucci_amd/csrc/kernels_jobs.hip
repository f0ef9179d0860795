// Mixed-size batched jobs in one persistent launch.
//
// The reference meshes each octree leaf as an independent thread-pool job
// (src/mesh/mod.rs:129-161).  Here a batch of independent grid jobs -- each
// with its own size n^3, power and iteration cap -- is one index space: the
// jobs' grids are concatenated, every wave of the persistent lane-refill loop
// finds its window's job by a search of the job offsets (kept in LDS), and its
// lanes evaluate distance plus the forward-mode (tangent) gradient for the
// unit normal.  A job's completion time is the latest wall-clock stamp of its
// points' write-back (one atomicMax per wave and run of a job), so per-job
// latency comes out of the same launch.  The launch (plus its small reset
// kernel) can be captured in a hipGraph and replayed.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "internal.h"
#include "launch.h"
#include "point_sources.h"
#include "tangent.h"
#include "work_loop.h"

namespace cth {

struct JobDev {
    float start[3];
    float across[3];
    float divisor, inv;  // inv != 0 when divisor is a power of two
    float power;
    uint32_t max_iters;
    FastDiv n, n2;
    uint32_t offset;
};

constexpr int kMaxJobs = 1024;

__global__ void k_jobs_reset(unsigned long long* done, uint32_t njobs, unsigned long long* start) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < njobs) done[i] = 0ull;
    if (i == 0) *start = ~0ull;
}

constexpr uint32_t kNoJob = ~0u;

// One lane of the wave raises the job's completion stamp.
__device__ __forceinline__ void stamp_job(unsigned long long* done, uint32_t job, unsigned long long stamp) {
    if (job != kNoJob && (int)__lane_id() == __ffsll((unsigned long long)wave_mask(true)) - 1)
        atomicMax(done + job, stamp);
}

template <class Ev>
__global__ __launch_bounds__(256) void k_jobs(const JobDev* __restrict__ jobs, uint32_t njobs, MandelUniform u,
                                              float* __restrict__ dists, float* __restrict__ normals,
                                              unsigned long long* __restrict__ done, unsigned long long* start,
                                              WorkQueue q) {
    __shared__ uint32_t offs[kMaxJobs + 1];
    for (uint32_t i = threadIdx.x; i <= njobs; i += blockDim.x) offs[i] = (i < njobs) ? jobs[i].offset : q.total;
    __syncthreads();
    if (threadIdx.x == 0) atomicMin(start, (unsigned long long)wall_clock64());

    Ev ev;
    // live / holding lanes as wave-uniform lane masks (see refill_loop)
    const uint64_t wave = wave_mask(true);
    uint64_t live_m = 0, hold_m = 0;
    uint64_t capd_m = 0;  // held lanes whose point stopped at its job's iteration cap
    uint32_t idx = 0, job = 0, kcap = 1;
    // The wave's body count, and per lane the tick of its point's last body
    // (the job's cap counted from the tick at which the lane took the point).
    uint32_t tick = 0, tcap = 0;
    // The wave's latest write-back of job `sjob`.  It reaches the job's stamp
    // when the wave writes points of another job, and at the end: an atomic per
    // refill meets those of every wave in the same job on one address, and 18.4 M
    // points in 24 jobs then took 3.85 ms (2.27 so).
    uint32_t sjob = kNoJob;
    // The job of the window's next index and the first index after that job:
    // lanes take points of one job at a time, so that its description comes
    // through scalar loads (per lane: a search and 13 gathered words a refill).
    uint32_t wjob = 0, wend = 0;
    unsigned long long stamp = 0;
    float r = idle_start(ev, u);
    Window win;
    SinkGrad sink{dists, normals, nullptr, nullptr, nullptr, 0u};

    for (;;) {
        do {
            // write back held points and note the time for their jobs
            // SinkGrad reads k only as k == max_iters (the point stopped at the cap).
            if (__builtin_amdgcn_inverse_ballot_w64(hold_m)) {
                sink.max_iters = kcap;
                sink.put(idx, ev.finish(r), __builtin_amdgcn_inverse_ballot_w64(capd_m) ? kcap : 0u, r, ev.dr, ev);
            }
            uint64_t pend = hold_m;
            if (pend) {
                const unsigned long long now = wall_clock64();
                while (pend) {
                    const int lead = __ffsll((unsigned long long)pend) - 1;
                    const uint32_t jl = (uint32_t)__builtin_amdgcn_readlane((int)job, lead);
                    if (jl != sjob) {
                        stamp_job(done, sjob, stamp);
                        sjob = jl;
                    }
                    stamp = now;
                    pend &= ~wave_mask(job == jl);
                }
            }
            hold_m = 0;
            capd_m = 0;
            // a point that bails before its first body is held (see refill_loop)
            uint64_t need = wave & ~live_m;
            while (need != 0) {
                if (win.next >= win.end && !next_chunk(q, win)) break;
                if (win.next >= wend) {
                    // the last offset <= the index (a wave's chunks ascend)
                    uint32_t hi = njobs;
                    while (hi - wjob > 1) {
                        const uint32_t mid = (wjob + hi) >> 1;
                        if ((uint32_t)__builtin_amdgcn_readfirstlane((int)offs[mid]) <= win.next) wjob = mid; else hi = mid;
                    }
                    wend = (uint32_t)__builtin_amdgcn_readfirstlane((int)offs[wjob + 1]);
                }
                const JobDev& J = jobs[wjob];
                const uint32_t avail = (win.end < wend ? win.end : wend) - win.next;
                const uint32_t nneed = (uint32_t)__popcll(need);
                const uint32_t rank = lane_rank(need);
                const bool take = __builtin_amdgcn_inverse_ballot_w64(need) && rank < avail;
                if (take) {
                    idx = win.next + rank;
                    job = wjob;
                    uint32_t local = idx - J.offset;
                    uint32_t i = fdiv(local, J.n2);
                    uint32_t rem = local - i * J.n2.d;
                    uint32_t j = fdiv(rem, J.n);
                    uint32_t kk = rem - j * J.n.d;
                    uint32_t ijk[3] = {i, j, kk};
                    float c[3];
#pragma unroll
                    for (int a = 0; a < 3; ++a) {
                        float v = (J.inv != 0.0f) ? (float)ijk[a] * J.inv : div_rn((float)ijk[a], J.divisor);
                        c[a] = J.start[a] + J.across[a] * v;
                    }
                    kcap = J.max_iters;
                    tcap = tick + kcap - 1u;
                    ev.start(c[0], c[1], c[2], J.power, u);
                    r = ev.mag();
                }
                const uint64_t took = wave_mask(take);
                const uint64_t bailed = wave_mask(r > u.bailout) & took;
                hold_m |= bailed;
                live_m |= took & ~bailed;
                need &= ~took;
                win.next += (nneed < avail) ? nneed : avail;
            }
        } while (live_m == 0 && hold_m != 0);
        if (live_m == 0) break;
        const uint32_t limit = 64u - win.refill_at(q);
        do {
            const uint64_t cap_m = wave_mask(tcap == tick) & live_m;
            const float rn = tick_full(ev, r, u, live_m, cap_m);
            ++tick;
            const uint64_t bail_m = wave_mask(rn > u.bailout) & live_m & ~cap_m;
            live_m &= ~(cap_m | bail_m);
            hold_m |= cap_m | bail_m;
            capd_m |= cap_m;
        } while ((uint32_t)__popcll(live_m) > limit);
    }
    stamp_job(done, sjob, stamp);
    if (q.dynamic) wave_retire(q);
}

struct JobSet {
    int kind;
    float bailout;
    uint32_t njobs = 0;
    uint32_t total = 0;
    JobDev* dev = nullptr;
    std::vector<uint32_t> offsets;
};

static bool pow2_inv(float v, float& inv) {
    int e = 0;
    float m = frexpf(v, &e);
    inv = (v > 0.0f && m == 0.5f) ? ldexpf(1.0f, 1 - e) : 0.0f;
    return inv != 0.0f;
}

int jobs_prepare(Ctx&, int kind, float bailout, const cth_job* jobs, uint32_t njobs, JobSet** out) {
    if (njobs == 0 || njobs > kMaxJobs) return fail(CTH_E_INVALID, "job count must be in [1, 1024]");
    if (kind != CTH_SHAPE_MANDELBULB && kind != CTH_SHAPE_MANDELBULB_TRIG)
        return fail(CTH_E_INVALID, "jobs need a Mandelbulb kind");
    std::vector<JobDev> h(njobs);
    uint64_t off = 0;
    JobSet* js = new JobSet();
    js->kind = kind;
    js->bailout = bailout;
    for (uint32_t i = 0; i < njobs; ++i) {
        const cth_job& j = jobs[i];
        if (j.n == 0 || j.max_iters == 0 || !(j.divisor > 0.0f)) {
            delete js;
            return fail(CTH_E_INVALID, "job with n == 0, max_iters == 0 or divisor <= 0");
        }
        if (kind == CTH_SHAPE_MANDELBULB && (j.power != 8.0f)) {
            delete js;
            return fail(CTH_E_INVALID, "CTH_SHAPE_MANDELBULB jobs run the P8 polynomial: power must be 8");
        }
        JobDev& d = h[i];
        for (int a = 0; a < 3; ++a) {
            d.start[a] = j.start[a];
            d.across[a] = j.end[a] - j.start[a];
        }
        d.divisor = j.divisor;
        pow2_inv(j.divisor, d.inv);
        d.power = j.power;
        d.max_iters = j.max_iters;
        d.n = make_fastdiv(j.n);
        d.n2 = make_fastdiv(j.n * j.n);
        d.offset = (uint32_t)off;
        js->offsets.push_back((uint32_t)off);
        off += (uint64_t)j.n * j.n * j.n;
        if (off >= (1ull << 31)) {
            delete js;
            return fail(CTH_E_INVALID, "jobs exceed 2^31 points");
        }
    }
    js->njobs = njobs;
    js->total = (uint32_t)off;
    int rc = check_hip(hipMalloc((void**)&js->dev, njobs * sizeof(JobDev)), "hipMalloc jobs");
    if (!rc) rc = check_hip(hipMemcpy(js->dev, h.data(), njobs * sizeof(JobDev), hipMemcpyHostToDevice), "H2D jobs");
    if (rc) {
        if (js->dev) (void)hipFree(js->dev);
        delete js;
        return rc;
    }
    *out = js;
    return CTH_OK;
}

void jobs_destroy(JobSet* js) {
    if (!js) return;
    if (js->dev) (void)hipFree(js->dev);
    delete js;
}

uint32_t jobs_total(const JobSet* js) { return js ? js->total : 0; }
uint32_t jobs_offset(const JobSet* js, uint32_t i) { return (js && i < js->njobs) ? js->offsets[i] : 0; }

int jobs_run(Ctx& c, const JobSet& js, float* dists, float* normals, unsigned long long* done,
             unsigned long long* start, hipStream_t st) {
    MandelUniform u{};
    u.max_iters = 0;  // per job
    u.bailout = js.bailout;
    u.power = kPointPower;
    u.integral = (js.kind == CTH_SHAPE_MANDELBULB) ? 1 : 0;
    u.ipower = 8;
    hipLaunchKernelGGL(k_jobs_reset, dim3((js.njobs + 255) / 256), dim3(256), 0, st, done, js.njobs, start);
    int rc = check_hip(hipGetLastError(), "jobs reset launch");
    if (rc) return rc;
    uint32_t blocks = 0;
    WorkQueue q = make_queue(c, js.total, c.shape_jobs,
                             js.kind == CTH_SHAPE_MANDELBULB ? P8Tangent::kSpread : TrigNormal::kSpread, blocks, st);
    if (js.kind == CTH_SHAPE_MANDELBULB)
        hipLaunchKernelGGL((k_jobs<P8Tangent>), dim3(blocks), dim3(c.shape_jobs.block), 0, st, js.dev, js.njobs, u,
                           dists, normals, done, start, q);
    else
        hipLaunchKernelGGL((k_jobs<TrigNormal>), dim3(blocks), dim3(c.shape_jobs.block), 0, st, js.dev, js.njobs, u,
                           dists, normals, done, start, q);
    return check_hip(hipGetLastError(), "jobs launch");
}

}  // namespace cth
