"""Work counters of the refill kernels and the split surface-nets vertex pass."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu
F32 = np.float32


def test_work_counters_match_iteration_counts(ctx, torch_cuda):
    """The counters a span-sampling launch adds equal what its iteration
    output implies: loop bodies = sum of the per-corner counts, bailed
    evaluations = corners below the cap, evaluations = corners.  A trace
    launch counts one evaluation per ray step."""
    import cantucci_amd as ca
    from cantucci_amd import device as dev
    from test_gpu_de import octree_leaf_sample
    torch = torch_cuda
    shape = ca.Mandelbulb.classic(15, 2.0, ctx=ctx)
    spans = torch.from_numpy(octree_leaf_sample(500)).cuda()
    cnt = torch.zeros(3, dtype=torch.int64, device="cuda")
    ctx.count_work(cnt)
    try:
        _, _, it = dev.sample_spans(shape, spans, 8, with_cross=False, with_iters=True)
        torch.cuda.synchronize()
        bodies, bails, evals = (int(v) for v in cnt.cpu())
        it = it.cpu().numpy().astype(np.int64)
        assert bodies == int(it.sum()) and evals == it.size and bails == int((it < 15).sum())
        cnt.zero_()
        from cantucci_amd.workloads import orbit_poses
        cams = torch.from_numpy(orbit_poses(2, seed=0, W=40, H=24)).cuda()
        _, steps = dev.render_depth(shape, cams, 40, 24)
        torch.cuda.synchronize()
        assert int(cnt[2]) == int(steps.to(torch.int64).sum())
        assert 0 < int(cnt[1]) <= int(cnt[2]) and int(cnt[0]) > 0
    finally:
        ctx.count_work(None)
    # counting off: the counters stay as they are
    before = cnt.clone()
    dev.sample_spans(shape, spans, 8, with_cross=False)
    torch.cuda.synchronize()
    assert torch.equal(cnt, before)


@pytest.mark.parametrize("normals", ["fd6", "tangent"])
def test_deferred_emit_then_vertex_pass(ctx, torch_cuda, normals):
    """cth_mesh_emit_dev with deferred normals followed by
    cth_mesh_vertices_dev gives the records of the one-call emit bit for bit;
    the deferred records hold the leaf's 6-tap half-steps
    0.7 (e' - s') / res (src/mesh/buffer.rs:256) and a zero distance."""
    import cantucci_amd as ca
    from cantucci_amd import device as dev
    from test_gpu_de import octree_leaf_sample
    torch = torch_cuda
    shape = ca.Mandelbulb.classic(15, 2.0, ctx=ctx)
    spans = torch.from_numpy(octree_leaf_sample(300, seed=3)).cuda()
    d, _ = dev.sample_spans(shape, spans, 8, with_cross=False)
    _, _, v_ref, i_ref = dev.mesh(shape, spans, d, 8, normals)
    _, _, v_def, i_def = dev.mesh(shape, spans, d, 8, "deferred")
    v_def = v_def.clone()
    torch.cuda.synchronize()
    vd = v_def.cpu().numpy()
    assert torch.equal(i_ref, i_def)
    assert (vd[:, 6] == 0).all()
    assert np.array_equal(vd[:, :3].view(np.uint32), v_ref.cpu().numpy()[:, :3].view(np.uint32))
    # half-steps of every leaf: (0.7 * (e' - s')) / res in f32, e', s' the adjusted span
    sp = spans.cpu().numpy()
    of = (sp[:, 3:] - sp[:, :3]) / F32(8)
    s2, e2 = sp[:, :3] + -of, sp[:, 3:] + of
    hs = (F32(0.7) * (e2 - s2)) / F32(8)
    assert np.isin(vd[:, 3:6].view(np.uint32), hs.view(np.uint32)).all()
    dev.mesh_vertices(shape, v_def, normals)
    torch.cuda.synchronize()
    assert np.array_equal(v_def.cpu().numpy().view(np.uint32), v_ref.cpu().numpy().view(np.uint32))
    with pytest.raises(ca.CthError):
        dev.mesh_vertices(shape, v_def, "deferred")


@pytest.mark.parametrize("min_depth,max_depth", [(0, 0), (1, 0), (0, 1), (2, 3), (2, 5), (4, 4), (5, 5), (0, 6)])
@pytest.mark.parametrize("kind", ["p8", "trig", "sphere"])
def test_refinement_top_matches_levels(ctx, torch_cuda, kind, min_depth, max_depth):
    """The tree's top is refined in one launch, counted refinement level by
    level through the work loops: the same leaves and level counts for trees
    that end in the top, leave it at any level (forced splits included) or
    have nothing to refine, and for an output that holds only some leaves."""
    import cantucci_amd as ca
    from cantucci_amd import device as dev
    from cantucci_amd.workloads import half_diagonals
    torch = torch_cuda
    shape = {"p8": lambda: ca.Mandelbulb.classic(15, 2.0, ctx=ctx),
             "trig": lambda: ca.MandelbulbTrig(9, 2.0, 6.5, ctx=ctx),
             "sphere": lambda: ca.Sphere((0.1, 0.0, -0.2), 0.9, ctx=ctx)}[kind]()
    for root in ((-1.5,) * 3 + (1.5,) * 3, (4.0,) * 3 + (4.5,) * 3):
        hd = half_diagonals(root[3] - root[0], max_depth)
        cnt = torch.zeros(4, dtype=torch.int64, device="cuda")
        ctx.count_work(cnt)
        try:
            want, want_lc = dev.refine(shape, root, min_depth, max_depth, hd)
            torch.cuda.synchronize()
        finally:
            ctx.count_work(None)
        got, lc = dev.refine(shape, root, min_depth, max_depth, hd)
        assert (lc == want_lc).all()
        assert torch.equal(got, want)
        few = torch.full((max(1, want.shape[0] // 2) + 1, 6), 7.0, device="cuda")
        keep = few[:-1]
        dev.refine(shape, root, min_depth, max_depth, hd, leaves=keep)
        m = min(keep.shape[0], want.shape[0])
        assert torch.equal(keep[:m], want[:m])
        assert (few[-1] == 7.0).all()


@pytest.mark.parametrize("iters", [128, 129, 300])
@pytest.mark.parametrize("kind", ["p8", "p5", "real"])
def test_refinement_at_large_caps(ctx, torch_cuda, kind, iters):
    """Iteration caps on both sides of the one up to which the tree's top is one
    launch for every map: the counted refinement's leaves and level counts."""
    import cantucci_amd as ca
    from cantucci_amd import device as dev
    from cantucci_amd.workloads import half_diagonals
    torch = torch_cuda
    shape = {"p8": lambda: ca.Mandelbulb.classic(iters, 2.0, ctx=ctx),
             "p5": lambda: ca.Mandelbulb(iters, 2.0, 5, ctx=ctx),
             "real": lambda: ca.MandelbulbTrig(iters, 2.0, 6.5, ctx=ctx)}[kind]()
    root, hd = (-1.5,) * 3 + (1.5,) * 3, half_diagonals(3.0, 5)
    cnt = torch.zeros(4, dtype=torch.int64, device="cuda")
    ctx.count_work(cnt)
    try:
        want, want_lc = dev.refine(shape, root, 1, 5, hd)
        torch.cuda.synchronize()
    finally:
        ctx.count_work(None)
    got, lc = dev.refine(shape, root, 1, 5, hd)
    assert (lc == want_lc).all()
    assert torch.equal(got, want)


@pytest.mark.parametrize("iters", [1, 28, 29, 64, 65, 512, 513])
@pytest.mark.parametrize("kind", ["p8", "real", "sphere"])
def test_refinement_hands_over_at_any_level(ctx, torch_cuda, kind, iters):
    """The one workgroup hands over to the levels' own launches earlier the longer
    the evaluations are: leaves and level counts are the counted refinement's on
    both sides of each cap, from single levels to trees beyond its largest."""
    import cantucci_amd as ca
    from cantucci_amd import device as dev
    from cantucci_amd.workloads import half_diagonals
    torch = torch_cuda
    shape = {"p8": lambda: ca.Mandelbulb.classic(iters, 2.0, ctx=ctx),
             "real": lambda: ca.MandelbulbTrig(iters, 2.0, 6.5, ctx=ctx),
             "sphere": lambda: ca.Sphere((0.0, 0.1, 0.2), 0.9, ctx=ctx)}[kind]()
    root = (-1.5,) * 3 + (1.5,) * 3
    for mind, d in ((0, 0), (0, 3), (2, 2), (2, 3), (3, 5), (4, 4)):
        hd = half_diagonals(3.0, d)
        cnt = torch.zeros(4, dtype=torch.int64, device="cuda")
        ctx.count_work(cnt)
        try:
            want, want_lc = dev.refine(shape, root, mind, d, hd)
            torch.cuda.synchronize()
        finally:
            ctx.count_work(None)
        got, lc = dev.refine(shape, root, mind, d, hd)
        assert (lc == want_lc).all()
        assert torch.equal(got, want)
