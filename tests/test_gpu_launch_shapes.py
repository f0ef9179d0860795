"""Results do not depend on the launch shape.  Every persistent kernel family
(points and grids, span sampling, the mesh's vertex taps, tracing, gradients,
jobs) runs under extreme launch shapes and must give outputs bit-identical to
those of the default shapes:

* one 64-thread workgroup per CU, chunks of 64 indices, refill at 1 idle lane;
* 32 workgroups of 256 threads per CU (more than fit at once: the rest run
  after the first ones leave), chunks of 4096, refill only when all 64 lanes
  are idle;
* a static interleave with 128-thread workgroups and an odd threshold of 17.

What changes between shapes is the work queue, the refill events and the
lane bookkeeping, never a point's arithmetic."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [
    dict(block=64, blocks_per_cu=1, chunk=64, refill_min=1, dynamic=1),
    dict(block=256, blocks_per_cu=32, chunk=4096, refill_min=64, dynamic=1),
    dict(block=128, blocks_per_cu=4, chunk=256, refill_min=17, dynamic=0),
    dict(block=256, blocks_per_cu=16, chunk=64, refill_min=64, dynamic=0),
]


def _run_all(torch, ctx):
    """Every family's outputs on small seeded inputs, as host arrays."""
    import cantucci_amd as ca
    from cantucci_amd import _lib
    from cantucci_amd import device as dev
    from cantucci_amd import workloads as wl
    from test_gpu_mesh import octree_leaves
    out = {}
    p8 = ca.Mandelbulb.classic(15, 2.0, ctx=ctx)
    trig = ca.MandelbulbTrig(15, 2.0, 7.5, ctx=ctx)
    rng = np.random.default_rng(21)
    pts = torch.from_numpy(rng.uniform(-1.3, 1.3, (50000, 3)).astype(np.float32)).cuda()
    out["p8_d"], out["p8_it"] = dev.de_points(p8, pts, with_iters=True)
    out["trig_d"] = dev.de_points(trig, pts)
    out["grid"] = dev.de_grid(p8, (-1.5,) * 3, (1.5,) * 3, 32, 31.0)
    leaves = torch.from_numpy(np.ascontiguousarray(octree_leaves(1000, seed=5))).cuda()
    dists, cross = dev.sample_spans(p8, leaves, 8)
    out["dists"], out["cross"] = dists, cross
    out["voff"], out["ioff"], out["verts"], out["idx"] = dev.mesh(p8, leaves, dists, 8, "fd6")
    cams = torch.from_numpy(wl.orbit_poses(2, 3, 160, 90, 60.0)).cuda()
    out["depth"], out["steps"] = dev.render_depth(p8, cams, 160, 90)
    sp, sw = wl.shell_points(20000, 4)
    sp, sw = torch.from_numpy(sp).cuda(), torch.from_numpy(sw).cuda()
    out["tan_d"], out["tan_n"] = dev.normals(trig, sp, sw)
    out["vjp_d"], out["vjp_g"] = dev.de_vjp(trig, sp, sw)
    out["grad_d"], out["grad_g"] = dev.de_grad(trig, sp, sw)
    jobs = [dict(n=n, power=p, max_iters=c) for n, p, c in ((9, 2.5, 15), (16, 7.25, 8), (12, 11.5, 30))]
    js = dev.JobSet(ctx, _lib.CTH_SHAPE_MANDELBULB_TRIG, 2.0, jobs)
    jd = torch.empty(js.total, device="cuda")
    jn = torch.empty((js.total, 3), device="cuda")
    js.run(jd, jn, torch.zeros(js.njobs, dtype=torch.int64, device="cuda"),
           torch.zeros(1, dtype=torch.int64, device="cuda"))
    out["jobs_d"], out["jobs_n"] = jd, jn
    torch.cuda.synchronize()
    js.close()
    return {k: v.cpu().numpy() for k, v in out.items()}


def _bits(a):
    a = np.ascontiguousarray(a)
    return a.view(np.uint8) if a.dtype.itemsize == 1 else a.view(f"u{a.dtype.itemsize}")


def test_outputs_do_not_depend_on_launch_shape(torch_cuda):
    import cantucci_amd as ca
    from cantucci_amd import _lib
    torch = torch_cuda
    families = (_lib.CTH_KERNEL_DE, _lib.CTH_KERNEL_TRACE, _lib.CTH_KERNEL_ADJOINT, _lib.CTH_KERNEL_SPANS,
                _lib.CTH_KERNEL_JOBS, _lib.CTH_KERNEL_MESH)
    ctx = ca.Context(0, "parity")
    try:
        base = _run_all(torch, ctx)
        for shape in SHAPES:
            for f in families:
                ctx.set_launch(f, **shape)
            got = _run_all(torch, ctx)
            for k in base:
                assert got[k].shape == base[k].shape, (shape, k)
                assert (_bits(got[k]) == _bits(base[k])).all(), f"{k} differs under {shape}"
            print(f"{shape}: all {len(base)} outputs bit-identical")
    finally:
        ctx.close()


@pytest.mark.parametrize("off", [-1, 0, 1])
@pytest.mark.parametrize("what", ["normals", "render"])
def test_large_default_launches_claim(torch_cuda, what, off):
    """Default static shapes claim their chunks from 8 chunks of 64 indices for
    each resident wave on (16 waves per CU for the tangent normals, 32 for the
    trace): below, at and beyond that size the outputs are those of a static
    shape given by the caller; at it, also when the launch is captured into a
    graph that has no counters of its own, over several replays with claiming
    launches in between."""
    import cantucci_amd as ca
    from cantucci_amd import _lib
    from cantucci_amd import device as dev
    from cantucci_amd import workloads as wl
    torch = torch_cuda
    auto, static = ca.Context(0, "parity"), ca.Context(0, "parity")
    try:
        for f in (_lib.CTH_KERNEL_TRACE, _lib.CTH_KERNEL_ADJOINT):
            static.set_launch(f, 256, 16, 256, 32, dynamic=0)
        cus = torch.cuda.get_device_properties(0).multi_processor_count
        if what == "render":
            W, H = 2048, 8 * 64 * 32 * cus // 2048 + off
            cams = torch.from_numpy(wl.orbit_poses(1, 2, W, H)).cuda()
            bufs = (torch.empty((1, H, W), device="cuda"), torch.empty((1, H, W), dtype=torch.int32, device="cuda"))

            def run(c):
                dev.render_depth(ca.Mandelbulb.classic(4, 2.0, ctx=c), cams, W, H, max_steps=12,
                                 depth=bufs[0], steps=bufs[1])
        else:
            n = 8 * 64 * 16 * cus + 65 * off
            pts = torch.rand((n, 3), device="cuda", generator=torch.Generator(device="cuda").manual_seed(7))
            bufs = (torch.empty(n, device="cuda"), torch.empty((n, 3), device="cuda"))

            def run(c):
                dev.normals(ca.Mandelbulb.classic(6, 2.0, ctx=c), pts, out=bufs[1], d=bufs[0])

        def result(f):
            for b in bufs:
                b.fill_(-1)
            f()
            torch.cuda.synchronize()
            return [b.view(torch.int32).clone() for b in bufs]

        def check(f):
            return all(torch.equal(x, y) for x, y in zip(want, result(f)))

        want = result(lambda: run(static))
        assert check(lambda: run(auto))
        if off == 0:
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g):
                run(auto)
            for _ in range(3):
                assert check(g.replay)
                assert check(lambda: run(auto))
    finally:
        auto.close()
        static.close()


@pytest.mark.parametrize("waves", [16, 17, 18, 20, 24, 25])
@pytest.mark.parametrize("what", ["points", "normals"])
def test_middle_launches_grow(torch_cuda, what, waves):
    """Launches of the trig map and the tangents grow by whole workgroups per CU
    from 8/3 chunks of 64 for each of their first waves on: point counts that
    give 3/8 wave a chunk on both sides of each step, one point short of and
    beyond a chunk, against a dense launch shape given by the caller."""
    import cantucci_amd as ca
    from cantucci_amd import _lib
    from cantucci_amd import device as dev
    torch = torch_cuda
    auto, given = ca.Context(0, "parity"), ca.Context(0, "parity")
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    w = waves if what == "points" else waves - 8
    try:
        for f in (_lib.CTH_KERNEL_DE, _lib.CTH_KERNEL_ADJOINT):
            given.set_launch(f, 256, 4, 64, 64, dynamic=1)
        for off in (-1, 1):
            n = 64 * cus * w * 8 // 3 + off
            gen = torch.Generator(device="cuda").manual_seed(waves)
            pts = torch.rand((n, 3), device="cuda", generator=gen) * 2.4 - 1.2
            outs = []
            for c in (auto, given):
                shape = ca.Mandelbulb(5, 2.0, 3, ctx=c)
                outs.append(dev.normals(shape, pts) if what == "normals" else (dev.de_points(shape, pts),))
            for a, b in zip(*outs):
                assert torch.equal(a.view(torch.int32), b.view(torch.int32))
    finally:
        auto.close()
        given.close()


def test_captures_without_counters(torch_cuda):
    """Contexts whose shapes claim (as recorded ones do), captured by torch, whose
    graphs have no counters: replays beside claiming launches on another stream
    give the eager outputs, and still do once the context is gone (the launches
    hold nothing of it)."""
    import cantucci_amd as ca
    from cantucci_amd import _lib
    from cantucci_amd import device as dev
    from cantucci_amd import workloads as wl
    torch = torch_cuda
    c, other = ca.Context(0, "parity"), ca.Context(0, "parity")
    for f in (_lib.CTH_KERNEL_DE, _lib.CTH_KERNEL_TRACE, _lib.CTH_KERNEL_ADJOINT, _lib.CTH_KERNEL_JOBS):
        c.set_launch(f, 256, 2, 256, 16, dynamic=1)
    m = ca.Mandelbulb.classic(6, 2.0, ctx=c)
    n = 1 << 20
    pts = torch.rand((n, 3), device="cuda", generator=torch.Generator(device="cuda").manual_seed(3)) * 2.4 - 1.2
    spans = torch.cat([pts[:2000] - 0.05, pts[:2000] + 0.05], 1).contiguous()
    cams = torch.from_numpy(wl.orbit_poses(1, 2, 1024, 512)).cuda()
    js = dev.JobSet(c, _lib.CTH_SHAPE_MANDELBULB, 2.0, [dict(n=40 + k, power=8.0, max_iters=5 + k) for k in range(6)])
    nrm, d = torch.empty((n, 3), device="cuda"), torch.empty(n, device="cuda")
    sd = torch.empty((2000, 729), device="cuda")
    depth, steps = torch.empty((1, 512, 1024), device="cuda"), torch.empty((1, 512, 1024), dtype=torch.int32,
                                                                           device="cuda")
    jd, jn = torch.empty(js.total, device="cuda"), torch.empty((js.total, 3), device="cuda")
    done = torch.zeros(js.njobs, dtype=torch.int64, device="cuda")
    start = torch.zeros(1, dtype=torch.int64, device="cuda")
    bufs = (nrm, d, sd, depth, steps, jd, jn)

    def work(shape):
        dev.normals(shape, pts, out=nrm, d=d)
        dev.sample_spans(shape, spans, 8, with_cross=False, out=sd)
        dev.render_depth(shape, cams, 1024, 512, max_steps=12, depth=depth, steps=steps)
        js.run(jd, jn, done, start)
        return dev.de_points(shape, pts), dev.de_grid(shape, (-1.2,) * 3, (1.2,) * 3, 96, 95.0)

    def result(f, outs):
        for b in bufs + outs:
            b.fill_(-1)
        f()
        torch.cuda.synchronize()
        return [b.view(torch.int32).clone() for b in bufs + outs]

    try:
        outs = work(m)
        torch.cuda.synchronize()
        want = [b.view(torch.int32).clone() for b in bufs + outs]
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            gouts = work(m)
        side = torch.cuda.Stream()
        o2 = ca.Mandelbulb.classic(6, 2.0, ctx=c)
        e = torch.empty_like(nrm)

        def beside():
            g.replay()
            with torch.cuda.stream(side):
                for _ in range(8):
                    dev.normals(o2, pts, out=e)

        for f in (g.replay, beside, beside):
            for a, b in zip(result(f, gouts), want):
                assert torch.equal(a, b)
        assert torch.equal(e.view(torch.int32), want[0])
        c.close()
        dev.normals(ca.Mandelbulb.classic(4, 2.0, ctx=other), pts)  # claims from its own ring
        for a, b in zip(result(g.replay, gouts), want):
            assert torch.equal(a, b)
    finally:
        torch.cuda.synchronize()
        js.close()
        c.close()
        other.close()


def test_shape_read_and_set_back(torch_cuda):
    """A family's shape can be read, replaced and set back: what it reports tells
    the default, whose large launches claim, from the same numbers set static."""
    import cantucci_amd as ca
    from cantucci_amd import _lib
    c = ca.Context(0, "parity")
    try:
        for f in (_lib.CTH_KERNEL_DE, _lib.CTH_KERNEL_TRACE, _lib.CTH_KERNEL_ADJOINT, _lib.CTH_KERNEL_SPANS,
                  _lib.CTH_KERNEL_JOBS, _lib.CTH_KERNEL_MESH):
            was = c.get_launch(f)
            assert was["dynamic"] == (1 if f in (_lib.CTH_KERNEL_SPANS, _lib.CTH_KERNEL_MESH) else 2)
            for dyn in (0, 1):
                c.set_launch(f, **{**was, "dynamic": dyn})
                assert c.get_launch(f) == {**was, "dynamic": dyn}
            c.set_launch(f, **was)
            assert c.get_launch(f) == was
    finally:
        c.close()
