"""The work that programs built on this framework have it do, as timed cases.

Every case goes through the package's public entry points: the host-side
mirrors of the reference's per-frame calls (one distance query, the focus
rays, one leaf's mesh), and the device-tensor calls of batch users (grids,
point batches, octree meshing, depth images, normals, gradients, job
batches).  Cases are plain dicts; "kind" picks the path and the other keys its
sizes and options:

  query     Shape.batch_min_distance_from on host points (n = 1: the fly
            camera's query of every frame)
  focii     get_focii: the focus rays of one frame, built and marched
  leaf      MeshBuffer.generate_for_box: one octree leaf meshed to host buffers
  app_mesh  the application's leaves (its bounding box split `levels` times)
            sampled and meshed on the device in one batch
  grid      distances on an n^3 grid
  points    distances of n scattered points, integer power
  octree    refinement to `depth`, span sampling and surface nets of every
            surface leaf
  render    sphere-traced depth images of orbit cameras
  normals   distances and unit normals of shell points, one power per point
            or the polynomial power 8
  fit       the distance op's forward pass and its gradients with respect to
            points and powers, by the named sweep
  jobs      a batch of grid jobs of mixed size, power and iteration cap

`octree`, `render`, `normals` and `jobs` use the launch shapes that the
package's tuner recorded for these workloads, as batch programs do; the
others run on a context's defaults, which is what the host mirrors use.

Mesh sizes depend on the sampled surface, so programs keep buffers with room
to spare for them (a renderer's vertex and index buffers, the octree's leaf and
distance arrays); what a pass returns of such a buffer is all of it.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import cantucci_amd as ca
from cantucci_amd import _lib, autotune
from cantucci_amd import device as dev
from cantucci_amd import workloads as wl
from cantucci_amd.mesh import MeshBuffer, create_spans, get_focii

# One P8 loop body is 75 operations; the mean number of bodies per evaluation
# depends on where a path samples (near the surface most orbits run long).
BODY_FLOP = 75.0
BODIES = {"query": 2.7, "grid": 2.7, "points": 2.7, "surface": 9.0, "shell": 4.0, "ray": 1.6, "jobs": 3.0}
# Forward and tangent (or reverse) work of a differentiated body, in bodies.
GRAD_BODIES = 4.0

APP_SHAPE = {"iters": 6, "bailout": 2.5}      # the application's Mandelbulb
BENCH_SHAPE = {"iters": 15, "bailout": 2.0}   # the benchmark workloads'


def listed():
    return [
        # The fly camera asks for one distance per frame: pure call latency.
        {"name": "query_one", "kind": "query", "n": 1, "power": 8, **APP_SHAPE},
        # A host program's batch through the Shape trait, points and distances in host memory.
        {"name": "query_batch", "kind": "query", "n": 100_003, "power": 8, **BENCH_SHAPE},
        # The 25 focus rays of a frame: a few long dependent chains.
        {"name": "focus_rays", "kind": "focii", "focus_points": 5, "power": 8, **APP_SHAPE},
        # One leaf's mesh job at the application's resolution, host buffers out.
        {"name": "leaf_mesh", "kind": "leaf", "res": 64, "power": 8, **APP_SHAPE},
        # The application's first update on the device: 64 leaves at resolution 64.
        {"name": "app_mesh", "kind": "app_mesh", "levels": 2, "res": 64, "power": 8, **APP_SHAPE},
        # The plain 64^3 grid: a small launch.
        {"name": "grid_64", "kind": "grid", "n": 64, "power": 8, **BENCH_SHAPE},
        # Scattered device points at another integer power (the generic map), a ragged count.
        {"name": "points_p5", "kind": "points", "n": 1_000_003, "power": 5, **BENCH_SHAPE},
        # Adaptive meshing: refinement, span sampling, surface nets, 6-tap normals.
        {"name": "octree_d7", "kind": "octree", "depth": 7, "res": 8, "power": 8, **BENCH_SHAPE},
        # Depth images for a set of poses.
        {"name": "render_8x1080p", "kind": "render", "width": 1920, "height": 1080, "poses": 8, "power": 8,
         **BENCH_SHAPE},
        # Normals of points near the surface, a real power per point.
        {"name": "normals_shell", "kind": "normals", "n": 1 << 21, "per_point": True, **BENCH_SHAPE},
        # One step of fitting points and powers: distances, then both gradients by the reverse sweep.
        {"name": "fit_reverse", "kind": "fit", "n": 300_001, "sweep": "reverse", "per_point": True, **BENCH_SHAPE},
        # Independent grid jobs of mixed sizes in one launch.
        {"name": "jobs_24", "kind": "jobs", "jobs": 24, "layout": 5, "bailout": 2.0},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["query", "focii", "leaf", "app_mesh", "grid", "points", "octree", "render", "normals", "fit",
                       "jobs"])
    shape = dict(rng.choice([APP_SHAPE, BENCH_SHAPE]))
    if kind == "query":
        return {"kind": kind, "n": _log_int(rng, 1, 300_000), "power": 8, **shape}
    if kind == "focii":
        return {"kind": kind, "focus_points": rng.randint(3, 24), "power": 8, **shape}
    if kind == "leaf":
        return {"kind": kind, "res": rng.choice([8, 16, 32, 64]), "power": 8, "iters": rng.randint(4, 16),
                "bailout": rng.choice([2.0, 2.5])}
    if kind == "app_mesh":
        return {"kind": kind, "levels": rng.randint(1, 2), "res": rng.choice([16, 32, 64]), "power": 8,
                "iters": rng.randint(4, 16), "bailout": rng.choice([2.0, 2.5])}
    if kind == "grid":
        return {"kind": kind, "n": _log_int(rng, 16, 256), "power": 8, **shape}
    if kind == "points":
        return {"kind": kind, "n": _log_int(rng, 1000, 2_000_000), "power": rng.choice([8, 8, 2, 3, 5, 7, 9]), **shape}
    if kind == "octree":
        return {"kind": kind, "depth": rng.randint(4, 6), "res": rng.choice([4, 8, 16]), "power": 8,
                "iters": rng.randint(6, 15), "bailout": 2.0}
    if kind == "render":
        return {"kind": kind, "width": _log_int(rng, 161, 1920), "height": _log_int(rng, 120, 1080),
                "poses": rng.randint(1, 8), "power": 8, **shape}
    if kind == "normals":
        return {"kind": kind, "n": _log_int(rng, 1000, 2_000_000), "per_point": rng.choice([True, False]), **shape}
    if kind == "fit":
        return {"kind": kind, "n": _log_int(rng, 1000, 300_000), "sweep": rng.choice(["forward", "reverse"]),
                "per_point": rng.choice([True, False]), **shape}
    return {"kind": kind, "jobs": rng.randint(3, 24), "layout": rng.randrange(1 << 16), "bailout": 2.0}


# Contexts are handles that a program keeps; one per workload serves every
# state, as calls on one context run one after another here.
_CTX = {}


def _context(tuned=()):
    if tuned not in _CTX:
        ctx = ca.Context(0, "parity")
        for name in tuned:
            autotune.apply(ctx, name)
        _CTX[tuned] = ctx
    return _CTX[tuned]


def _job_layout(case):
    return wl.mixed_jobs(jobs=case["jobs"], seed=case["layout"])


def _uniform(seed, n, lo, hi):
    return wl.uniform(seed * 1_000_003 + 17, n, lo, hi)


def _host_points(case, seed):
    return _uniform(seed, 3 * case["n"], -1.5, 1.5).reshape(-1, 3).astype(np.float32)


def _shell(case, seed):
    return wl.shell_points(case["n"], seed * 1_000_003 + 23)


def _grid_box(case, seed):
    off = _uniform(seed, 3, -0.02, 0.02)
    return [float(np.float32(v)) for v in -1.5 + off], [float(np.float32(v)) for v in 1.5 + off]


def _focus_camera(seed):
    # the application's projection; the eye on a sphere of radius 3, looking near the origin
    u = _uniform(seed, 6, 0.0, 1.0)
    cos_t, phi = 1.0 - 2.0 * (0.05 + 0.9 * u[0]), 2.0 * math.pi * u[1]
    sin_t = math.sqrt(1.0 - cos_t * cos_t)
    eye = 3.0 * np.array([sin_t * math.cos(phi), sin_t * math.sin(phi), cos_t])
    aim = 0.2 * (u[2:5] - 0.5) - eye
    return [float(v) for v in eye], [float(v) for v in aim]


def _octree_cap(depth):
    return int(1.3 * _octree_leaves(depth)) + 256


def _leaf_cap(res):
    return min(res ** 3, 16 * res * res)


def _mesh_into(st, nleaves, res):
    """Surface nets of the first `nleaves` leaves into the state's buffers,
    through the two device calls of the C interface."""
    shape, h = st["shape"], st["shape"].ctx.handle
    nv, ni = C.c_uint64(), C.c_uint64()
    stream = torch.cuda.current_stream().cuda_stream
    _lib.check(_lib.lib.cth_mesh_count_dev(h, st["dists"].data_ptr(), nleaves, res, st["voff"].data_ptr(),
                                           st["ioff"].data_ptr(), None, C.byref(nv), C.byref(ni), stream))
    if nv.value > st["verts"].shape[0] or ni.value > st["idx"].shape[0]:
        raise RuntimeError("mesh buffers too small")
    _lib.check(_lib.lib.cth_mesh_emit_dev(h, C.byref(shape.desc), st["leaves"].data_ptr(), st["dists"].data_ptr(),
                                          nleaves, res, _lib.CTH_NORMALS_FD6, st["voff"].data_ptr(),
                                          st["ioff"].data_ptr(), nv.value, st["verts"].data_ptr(),
                                          st["idx"].data_ptr(), stream))
    return nv.value, ni.value


def _job_offset(case, seed, i):
    return [float(np.float32(v)) for v in -1.5 + _uniform(seed * 131 + i, 3, -0.02, 0.02)]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "jobs":
        ctx = _context(("jobs",))
        N, P, cap = _job_layout(case)
        jobs = []
        for i, (n, p, c) in enumerate(zip(N, P, cap)):
            s = _job_offset(case, seed, i)
            jobs.append(dict(n=int(n), power=float(p), max_iters=int(c), start=s, end=[v + 3.0 for v in s]))
        js = dev.JobSet(ctx, _lib.CTH_SHAPE_MANDELBULB_TRIG, case["bailout"], jobs)
        return {"case": case, "jobs": js, "dists": torch.empty(js.total, device="cuda"),
                "normals": torch.empty((js.total, 3), device="cuda"),
                "done": torch.zeros(js.njobs, dtype=torch.int64, device="cuda"),
                "start": torch.zeros(1, dtype=torch.int64, device="cuda")}
    tuned = {"octree": ("spans", "mesh"), "render": ("trace",), "normals": ("tangent",)}.get(kind, ())
    ctx = _context(tuned)
    if case.get("per_point"):
        shape = ca.MandelbulbTrig(case["iters"], case["bailout"], 8.0, ctx=ctx)
    else:
        shape = ca.Mandelbulb(case["iters"], case["bailout"], case.get("power", 8), ctx=ctx)
    st = {"case": case, "shape": shape}
    if kind == "query":
        st["pts"] = _host_points(case, seed)
    elif kind == "focii":
        st["eye"], st["aim"] = _focus_camera(seed)
        st["hits"] = np.zeros((case["focus_points"] ** 2, 3), np.float32)
    elif kind == "leaf":
        # a leaf of the application's octree over its bounding box, which all hold surface near the middle
        spans = [c for a in create_spans(shape.bounding_box()) for c in create_spans(a)]
        st["span"] = spans[int(_uniform(seed, 1, 0, len(spans))[0])]
        off = _uniform(seed + 1, 3, -0.01, 0.01)
        st["span"] = tuple(tuple(float(np.float32(v + o)) for v, o in zip(corner, off)) for corner in st["span"])
        cap = _leaf_cap(case["res"])
        st["verts"], st["idx"] = np.zeros((cap, 7), np.float32), np.zeros(18 * cap, np.uint32)
    elif kind == "app_mesh":
        spans = [shape.bounding_box()]
        for _ in range(case["levels"]):
            spans = [c for a in spans for c in create_spans(a)]
        # the leaves in an order of their own, as splits and drops leave them
        spans = [spans[i] for i in np.argsort(_uniform(seed, len(spans), 0.0, 1.0))]
        st["spans"] = torch.tensor([[*a, *b] for a, b in spans], dtype=torch.float32, device="cuda")
    elif kind == "grid":
        st["lo"], st["hi"] = _grid_box(case, seed)
    elif kind == "points":
        st["pts"] = torch.from_numpy(_host_points(case, seed)).cuda()
    elif kind == "octree":
        lo, hi = _grid_box(case, seed)
        st["root"] = (*lo, *hi)
        st["half_diag"] = wl.half_diagonals(3.0, case["depth"])
        cap, res = _octree_cap(case["depth"]), case["res"]
        verts = int(cap * 1.6 * res * res)
        st["leaves"] = torch.zeros((cap, 6), device="cuda")
        st["dists"] = torch.zeros((cap, (res + 1) ** 3), device="cuda")
        st["voff"] = torch.zeros(cap + 1, dtype=torch.int64, device="cuda")
        st["ioff"] = torch.zeros(cap + 1, dtype=torch.int64, device="cuda")
        st["verts"] = torch.zeros((verts, 7), device="cuda")
        st["idx"] = torch.zeros(6 * verts, dtype=torch.int32, device="cuda")
    elif kind == "render":
        W, H, n = case["width"], case["height"], case["poses"]
        st["cams"] = torch.from_numpy(wl.orbit_poses(n, seed, W, H, 60.0)).cuda()
        st["depth"] = torch.empty((n, H, W), device="cuda")
        st["steps"] = torch.empty((n, H, W), dtype=torch.int32, device="cuda")
    else:  # normals, fit
        pts, powers = _shell(case, seed)
        st["pts"] = torch.from_numpy(pts).cuda()
        st["powers"] = torch.from_numpy(powers).cuda() if case["per_point"] else None
        if kind == "fit":
            st["grad"] = torch.from_numpy(_uniform(seed + 7, case["n"], -1.0, 1.0).astype(np.float32)).cuda()
            st["pts"].requires_grad_(True)
            if st["powers"] is not None:
                st["powers"].requires_grad_(True)
    return st


def run(st):
    case, kind = st["case"], st["case"]["kind"]
    if kind == "jobs":
        st["jobs"].run(st["dists"], st["normals"], st["done"], st["start"])
        return st["dists"], st["normals"]
    shape = st["shape"]
    if kind == "query":
        if case["n"] == 1:
            return shape.min_distance_from(st["pts"][0])
        return shape.batch_min_distance_from(st["pts"])
    if kind == "focii":
        hits = get_focii(shape, st["eye"], st["aim"], 1.0, 16 / 9, 0.00004, 10.0, case["focus_points"])
        st["hits"][:len(hits)] = hits
        return len(hits), st["hits"]
    if kind == "leaf":
        buf, _ = MeshBuffer.generate_for_box(st["span"], shape, case["res"])
        st["verts"][:len(buf.vertices)] = buf.vertices.view(np.float32).reshape(-1, 7)
        st["idx"][:len(buf.indices)] = buf.indices
        return len(buf.vertices), len(buf.indices), st["verts"], st["idx"]
    if kind == "app_mesh":
        dists, _ = dev.sample_spans(shape, st["spans"], case["res"], with_cross=False)
        return dev.mesh(shape, st["spans"], dists, case["res"], "fd6")
    if kind == "grid":
        return dev.de_grid(shape, st["lo"], st["hi"], case["n"], float(case["n"] - 1))
    if kind == "points":
        return dev.de_points(shape, st["pts"], with_iters=True)
    if kind == "octree":
        leaves, counts = dev.refine(shape, st["root"], 2, case["depth"], st["half_diag"], leaves=st["leaves"])
        n = leaves.shape[0]
        dev.sample_spans(shape, leaves, case["res"], with_cross=False, out=st["dists"][:n])
        nv, ni = _mesh_into(st, n, case["res"])
        return n, counts, nv, ni, st["leaves"], st["dists"], st["voff"], st["ioff"], st["verts"], st["idx"]
    if kind == "render":
        return dev.render_depth(shape, st["cams"], case["width"], case["height"], 256, 0.0, 1e-4, 10.0,
                                depth=st["depth"], steps=st["steps"])
    if kind == "normals":
        return dev.normals(shape, st["pts"], st["powers"])
    st["pts"].grad = None
    inputs = [st["pts"]]
    if st["powers"] is not None:
        inputs.append(st["powers"])
    d = dev.distance(shape, st["pts"], st["powers"], sweep=case["sweep"])
    return (d.detach(), *torch.autograd.grad(d, inputs, st["grad"]))


# Surface leaves of the octree workload by depth (about 5.5 times as many per
# level: the surface's dimension is a little over 2) and vertices per leaf.
def _octree_leaves(depth):
    return 921_604 * 5.5 ** (depth - 8)


def work(case):
    kind, body = case["kind"], BODY_FLOP
    if kind == "query":
        return {"bytes": 16 * case["n"], "flops": BODIES["query"] * body * case["n"]}
    if kind == "focii":
        n = case["focus_points"] ** 2
        return {"bytes": 12 * n + 40, "flops": 20 * 3 * body * n}
    if kind in ("leaf", "app_mesh"):
        leaves = 8 ** case["levels"] if kind == "app_mesh" else 1
        res = case["res"]
        corners, verts = leaves * (res + 1) ** 3, leaves * 2.5 * res * res
        return {"bytes": 24 * leaves + verts * (28 + 24), "flops": 4.0 * body * (corners + 7 * verts)}
    if kind == "grid":
        return {"bytes": 4 * case["n"] ** 3, "flops": BODIES["grid"] * body * case["n"] ** 3}
    if kind == "points":
        return {"bytes": 20 * case["n"], "flops": BODIES["points"] * body * case["n"]}
    if kind == "octree":
        leaves, res = _octree_leaves(case["depth"]), case["res"]
        corners, verts = leaves * (res + 1) ** 3, leaves * 80.0 * (res / 8) ** 2
        return {"bytes": 24 * leaves + 4 * corners + verts * (28 + 21),
                "flops": BODIES["surface"] * body * (corners + 7 * verts)}
    if kind == "render":
        n = case["width"] * case["height"] * case["poses"]
        return {"bytes": 8 * n, "flops": 13.2 * (BODIES["ray"] * body + 15) * n}
    if kind == "normals":
        n = case["n"]
        return {"bytes": n * (12 + 16 + (4 if case["per_point"] else 0)),
                "flops": GRAD_BODIES * BODIES["shell"] * body * n}
    if kind == "fit":
        n = case["n"]
        return {"bytes": n * (12 + 4 + 4 + 12 + (8 if case["per_point"] else 0)),
                "flops": (1 + GRAD_BODIES) * BODIES["shell"] * body * n}
    total = float(np.sum(_job_layout(case)[0].astype(np.float64) ** 3))
    return {"bytes": 16 * total, "flops": GRAD_BODIES * BODIES["jobs"] * body * total}


# ---------------------------------------------------------------------------
# The same values in 64 bits
# ---------------------------------------------------------------------------

def _rotate_p8(x, y, z):
    x2, y2, z2 = x * x, y * y, z * z
    x4, y4, z4 = x2 * x2, y2 * y2, z2 * z2
    x6, y6, z6 = x4 * x2, y4 * y2, z4 * z2
    w2 = x2 + y2
    w4 = w2 * w2
    a = 1 + (z4 * z4 - 28 * z6 * w2 + 70 * z4 * w4 - 28 * z2 * w2 * w4) / (w4 * w4)
    return (a * (x4 * x4 - 28 * x6 * y2 + 70 * x4 * y4 - 28 * x2 * y6 - y4 * y4),
            8 * a * x * y * (x6 - 7 * x4 * y2 + 7 * x2 * y4 - y6),
            8 * z * torch.sqrt(w2) * (z2 - w2) * (z4 - 6 * z2 * w2 + w4))


def _rotate_trig(x, y, z, r, power):
    th, ph = torch.acos(z / r) * power, torch.atan2(y, x) * power
    R = r ** power
    return torch.sin(th) * torch.cos(ph) * R, torch.sin(ph) * torch.sin(th) * R, torch.cos(th) * R


def _distance(pts, power, iters, bailout):
    """Distances of (n, 3) f64 points; power 8 (an int: the polynomial), another
    int or an (n,) tensor (the trigonometric map).  Differentiable."""
    n = pts.shape[0]
    at = torch.arange(n, device=pts.device)
    p = pts
    x, y, z = p.unbind(1)
    pw = power
    dr = torch.ones(n, dtype=torch.float64, device=pts.device)
    r = torch.sqrt(x * x + y * y + z * z)
    done = []
    for k in range(iters + 1):
        end = (r > bailout) if k < iters else torch.ones_like(r, dtype=torch.bool)
        done.append((at[end], r[end], dr[end]))
        go = ~end
        at, p, x, y, z, r, dr = at[go], p[go], x[go], y[go], z[go], r[go], dr[go]
        if torch.is_tensor(pw):
            pw = pw[go]
        if at.numel() == 0:
            break
        dr = r ** (pw - 1) * pw * dr + 1
        if k + 1 < iters:  # the last body's rotation is not read
            if not torch.is_tensor(pw) and pw == 8:
                x, y, z = _rotate_p8(x, y, z)
            else:
                x, y, z = _rotate_trig(x, y, z, r, pw)
            x, y, z = x + p[:, 0], y + p[:, 1], z + p[:, 2]
            r = torch.sqrt(x * x + y * y + z * z)
        else:
            done.append((at, r, dr))
            break
    order = torch.cat([d[0] for d in done])
    rf, drf = torch.cat([d[1] for d in done]), torch.cat([d[2] for d in done])
    out = 0.5 * torch.log(rf) * rf / drf
    return out[torch.argsort(order)]


def _in_parts(n, f, part=1 << 19):
    parts = [f(slice(i, min(n, i + part))) for i in range(0, n, part)]
    return [torch.cat(c) for c in zip(*parts)] if parts else []


def _with_grad(pts, power, iters, bailout, grad=None):
    """(d, dd/dp, dd/dpower or None), times `grad` where it is given."""
    def part(s):
        p = pts[s].detach().requires_grad_(True)
        tensor = torch.is_tensor(power)
        w = power[s].detach().requires_grad_(True) if tensor else power
        d = _distance(p, w, iters, bailout)
        g = torch.autograd.grad(d, [p, w] if tensor else [p], torch.ones_like(d) if grad is None else grad[s])
        return (d.detach(), *g)
    return _in_parts(pts.shape[0], part)


def _grid_points(lo, hi, n, divisor):
    """Grid points as the f32 sampling places them (they are inputs of the map)."""
    axes = []
    for a in range(3):
        s, e = np.float32(lo[a]), np.float32(hi[a])
        i = np.arange(n, dtype=np.float32) / np.float32(divisor)
        axes.append(torch.from_numpy((s + (e - s) * i).astype(np.float64)).cuda())
    return torch.stack(torch.meshgrid(*axes, indexing="ij"), -1).reshape(-1, 3)


def exact(case, seed):
    kind = case["kind"]
    # Meshes and marched rays: what is sampled next follows from the sign or
    # the step before, so these outputs have no 64-bit counterpart of one layout.
    if kind in ("focii", "leaf", "app_mesh", "octree", "render"):
        return None
    if kind == "jobs":
        d, g = [], []
        for i, (n, p, c) in enumerate(zip(*_job_layout(case))):
            s = _job_offset(case, seed, i)
            pts = _grid_points(s, [v + 3.0 for v in s], int(n), float(n - 1.0))
            p = float(p)
            w = torch.full((pts.shape[0],), p, dtype=torch.float64, device="cuda")
            d.append(_in_parts(pts.shape[0], lambda q: (_distance(pts[q], w[q], int(c), case["bailout"]),), 1 << 21)[0])
        # inside the set the normals' orbits are chaotic: most of a job's interior has no stable normal
        return torch.cat(d), None
    iters, bailout = case["iters"], case["bailout"]
    if kind in ("query", "points"):
        pts = torch.from_numpy(_host_points(case, seed)).cuda().double()
        d = _in_parts(case["n"], lambda s: (_distance(pts[s], case["power"], iters, bailout),), 1 << 20)[0]
        if kind == "points":
            return d, None
        return float(d[0]) if case["n"] == 1 else d
    if kind == "grid":
        lo, hi = _grid_box(case, seed)
        pts = _grid_points(lo, hi, case["n"], float(case["n"] - 1))
        return _in_parts(pts.shape[0], lambda s: (_distance(pts[s], case["power"], iters, bailout),), 1 << 21)[0]
    pts, powers = _shell(case, seed)
    pts = torch.from_numpy(pts).cuda().double()
    power = torch.from_numpy(powers).cuda().double() if case["per_point"] else 8
    if kind == "normals":
        d, g = _with_grad(pts, power, iters, bailout)[:2]
        return d, g / g.norm(dim=1, keepdim=True)
    grad = torch.from_numpy(_uniform(seed + 7, case["n"], -1.0, 1.0).astype(np.float32)).cuda().double()
    d, *g = _with_grad(pts, power, iters, bailout, grad)
    # the gradients' norm is that of the few chaotic points inside the set,
    # where f32 and f64 orbits part: only the distances have a value to hold to
    return (d, *[None] * len(g))
