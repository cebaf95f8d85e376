"""Performance cases of the framework: whole frames, batches of frames and the single stages a
program calls, each through the public entry points (particleisosurface_amd.capi).

A case is a dict of plain values. `listed()` gives the standing cases, `draw(rng)` one more of the
same ranges, `prepare(case, seed)` what a program holds before the call, `run(state)` one pass,
`work(case)` the bytes and operations a pass cannot do without, `exact(case, seed)` the 64-bit
values of the outputs that have some.

The particle sets are the synthetic workloads of the benchmark (dam break, sloshing tank, crown
splash, multi-body pour) with their lattices, jitter and spray, generated on the GPU.
"""
import ctypes as C
import math

import numpy as np
import torch

from particleisosurface_amd import capi

PREC = {"fp32": capi.FP32, "fp32k": capi.FP32_KAHAN, "fp64": capi.FP64}
QEF = {"off": capi.QEF_OFF, "float": capi.QEF_REFERENCE, "svd64": capi.QEF_SVD64}


# ---- particle sets -------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _uniform(g, shape, lo=0.0, hi=1.0):
    return lo + (hi - lo) * torch.rand(shape, generator=g, device="cuda", dtype=torch.float64)


def _normal(g, shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float64)


def _lattice(nx, ny, nz, s):
    a = [torch.arange(n, device="cuda", dtype=torch.float64) * s for n in (nx, ny, nz)]
    return torch.stack(torch.meshgrid(*a, indexing="ij"), -1).reshape(-1, 3)


def _jitter(g, p, r):
    return p + _uniform(g, p.shape, -0.1 * r, 0.1 * r)


def _dam_break(g, case):
    """Block [0,.3)x[0,.15)x[0,.3) and a droplet of radius .05 (14 k particles at r = .005)."""
    r = 0.005
    block = _lattice(30, 15, 30, 2 * r)
    ball = _lattice(31, 41, 31, 2 * r)
    c = torch.tensor([0.15, 0.30, 0.15], device="cuda", dtype=torch.float64)
    ball = ball[((ball - c) ** 2).sum(1) <= 0.05 ** 2 + 1e-12]
    return _jitter(g, torch.cat([block, ball]), r), r


def _tank_height(x, y, phase):
    return 0.2 + 0.03 * torch.sin(2 * math.pi * x + phase) * torch.cos(4 * math.pi * y)


def _tank(g, case, n=None):
    """Sloshing tank of about n particles with spray: half uniform in the air, half in clusters."""
    n = case["particles"] if n is None else n
    r = float(np.float32((0.0125 / n) ** (1.0 / 3.0)))
    s = 2 * r
    phase = 2 * math.pi * torch.rand(1, generator=g, device="cuda", dtype=torch.float64)
    p = _lattice(math.ceil(1.0 / s - 1e-9), math.ceil(0.5 / s - 1e-9), math.ceil(0.23 / s) + 1, s)
    p = _jitter(g, p[p[:, 2] < _tank_height(p[:, 0], p[:, 1], phase)], r)
    spray = max(int(round(10000 * n / 1.578e6)), 8)

    def air(k):
        xy = torch.stack([_uniform(g, (k,)), _uniform(g, (k,), 0, 0.5)], 1)
        lo = _tank_height(xy[:, 0], xy[:, 1], phase) + 4 * r
        return torch.cat([xy, (lo + (0.35 - lo) * _uniform(g, (k,)))[:, None]], 1)

    half = spray // 2
    centres = air(min(50, spray - half))
    pick = torch.arange(spray - half, device="cuda") % len(centres)
    return torch.cat([p, air(half), centres[pick] + 3 * r * _normal(g, (spray - half, 3))]), r


def _crown(g, case):
    """Crown splash, r = .001: a pool of `layers` layers, a crown sheet and 5000 droplets."""
    r = 0.001
    s = 2 * r
    top = case["layers"] * s
    parts = [_lattice(300, 300, case["layers"], s)]
    for layer in range(3):
        rho = 0.08 - layer * s
        nth = int(round(2 * math.pi * rho / s))
        th = torch.arange(nth, device="cuda", dtype=torch.float64) * (2 * math.pi / nth)
        nz = torch.floor((0.05 + 0.01 * torch.sin(12 * th)) / s).long() + 1
        k = torch.arange(int(nz.max()), device="cuda")
        i, kk = torch.nonzero(k[None, :] < nz[:, None], as_tuple=True)
        parts.append(torch.stack([0.3 + rho * torch.cos(th[i]), 0.3 + rho * torch.sin(th[i]), top + kk * s], 1))
    rad = 3 * r * torch.exp(0.5 * _normal(g, (5000,)).clamp(-3, 3))
    cen = torch.stack([_uniform(g, (5000,), 0.22, 0.38), _uniform(g, (5000,), 0.22, 0.38),
                       _uniform(g, (5000,), top + 0.07, top + 0.21)], 1)
    m = math.ceil(float(rad.max()) / s)
    a = torch.arange(-m, m + 1, device="cuda", dtype=torch.float64) * s
    off = torch.stack(torch.meshgrid(a, a, a, indexing="ij"), -1).reshape(-1, 3)
    o2 = (off ** 2).sum(1)
    for b in range(0, 5000, 500):
        i, j = torch.nonzero(o2[None, :] <= (rad[b:b + 500] ** 2)[:, None], as_tuple=True)
        parts.append(cen[b + i] + off[j])
    return _jitter(g, torch.cat(parts), r), r


def _pour(g, case):
    """Multi-body pour, r = .0005: a pool of `layers` layers, a jet and 200 k spray particles."""
    r = 0.0005
    s = 2 * r
    top = case["layers"] * s
    a = torch.arange(-20, 21, device="cuda", dtype=torch.float64) * s
    disk = torch.stack(torch.meshgrid(a, a, indexing="ij"), -1).reshape(-1, 2)
    disk = disk[(disk ** 2).sum(1) <= 0.02 ** 2] + 0.25
    z = top + torch.arange(300, device="cuda", dtype=torch.float64) * s
    jet = torch.cat([disk[None].expand(300, -1, -1), z[:, None, None].expand(-1, len(disk), 1)], 2).reshape(-1, 3)
    cen = torch.stack([_uniform(g, (2000,), 0, 0.5), _uniform(g, (2000,), 0, 0.5),
                       _uniform(g, (2000,), top + 0.01, top + 0.13)], 1)
    spray = cen.repeat_interleave(100, 0) + 2 * r * _normal(g, (200000, 3))
    return torch.cat([_jitter(g, torch.cat([_lattice(500, 500, case["layers"], s), jet]), r), spray]), r


SCENES = {"dam": _dam_break, "tank": _tank, "crown": _crown, "pour": _pour}


def _particles(case, seed):
    """(n, 3) float32 on the GPU, the radius, and the generator that made them."""
    g = _gen(seed)
    p, r = SCENES[case["scene"]](g, case)
    return p.float().contiguous(), r, g


def _count(case):
    """Particles of a case, about."""
    if case["scene"] == "dam":
        return 14015
    if case["scene"] == "tank":
        return case["particles"]
    if case["scene"] == "crown":
        return 90000 * case["layers"] + 240000
    return 250000 * case["layers"] + 577000


# ---- the cases -----------------------------------------------------------------------------
def listed():
    frame = dict(kind="frame", input="device", precision="fp32k", qef="off", ani=1, poly6=0, depth=0)
    points = dict(kind="points", ani=1, poly6=0)
    return [
        # one small frame of a preview or a parameter study, defaults of the library, host particles
        dict(frame, name="frame_dam_14k_fp32", scene="dam", input="host", precision="fp32"),
        # the plain method of the reference in double on a tank with spray
        dict(frame, name="frame_tank_400k_fp64", scene="tank", particles=400000, precision="fp64"),
        # the headline frame: crown splash, 4 M particles from a simulation on the same GPU
        dict(frame, name="frame_crown_4m_fp32k", scene="crown", layers=42),
        # the same splash over a shallow pool with the QEF vertex of TNode::NodeCalcNode
        dict(frame, name="frame_crown_1m_qef", scene="crown", layers=10, qef="svd64"),
        # a large production frame with a deep octree
        dict(frame, name="frame_pour_12m_fp32k", scene="pour", layers=46, depth=12),
        # a sequence of uneven frames read from files, meshed in one call
        dict(kind="batch", name="batch_6_tanks_fp32k", scene="tank", frames=6, smallest=50000, largest=1500000,
             precision="fp32k"),
        # a caller that samples the field now and then (a probe, a ray march step): latency
        dict(points, name="points_1k_grad_fp32", scene="dam", precision="fp32", points=1000, grad=1, fresh=0,
             order="shuffled"),
        # field and gradient at many points around the fluid, in no particular order
        dict(points, name="points_1m_grad_fp32k", scene="tank", particles=1600000, precision="fp32k", points=1000003,
             grad=1, fresh=0, order="shuffled"),
        # an evaluator set up on a new frame (grid, anisotropy) and read at points in scan order
        dict(points, name="evaluator_700k_fp64", scene="tank", particles=700000, precision="fp64", points=50001,
             grad=0, fresh=1, order="scan"),
        # the dense lattice of UniformGrid::Run for volume rendering
        dict(kind="lattice", name="lattice_tank_120k_fp32", scene="tank", particles=120000, precision="fp32", ani=1,
             poly6=0),
        # vertex placement for edges found by the caller's own extraction
        dict(kind="edges", name="edges_200k_fp32k", scene="tank", particles=800000, precision="fp32k", edges=200000),
        # neighbour lists for a solver or a surface tension term, device buffers in and out
        dict(kind="neighbors", name="neighbors_300k", scene="tank", particles=500000, queries=300007),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "batch", "points", "points", "lattice", "edges", "neighbors"])
    prec = rng.choice(["fp32", "fp32k", "fp32k", "fp64"])
    if kind == "frame":
        scene = rng.choice(["tank", "tank", "crown", "pour"])
        ani, poly6 = rng.choice([(1, 0), (1, 0), (1, 0), (1, 1), (0, 1)])
        c = dict(kind=kind, scene=scene, input=rng.choice(["device", "host"]), precision=prec,
                 qef=rng.choice(["off", "off", "off", "float", "svd64"]), ani=ani, poly6=poly6, depth=0)
        if scene == "tank":
            c["particles"] = _log_int(rng, 14000, 2500000)
        elif scene == "crown":
            c["layers"] = _log_int(rng, 4, 42)
        else:
            c.update(layers=_log_int(rng, 4, 40), depth=12, precision="fp32k", qef="off", ani=1, poly6=0)
        return c
    if kind == "batch":
        lo = _log_int(rng, 30000, 100000)
        return dict(kind=kind, scene="tank", frames=rng.randint(2, 8), smallest=lo,
                    largest=_log_int(rng, 3 * lo, 1500000), precision=prec)
    n = _log_int(rng, 14000, 2000000)
    if kind == "points":
        return dict(kind=kind, scene="tank", particles=n, precision=prec, points=_log_int(rng, 500, 1500000),
                    grad=rng.randint(0, 1), fresh=rng.choice([0, 0, 1]), order=rng.choice(["shuffled", "scan"]),
                    ani=1, poly6=rng.choice([0, 0, 0, 1]))
    if kind == "lattice":
        return dict(kind=kind, scene="tank", particles=_log_int(rng, 14000, 300000), precision=prec, ani=1,
                    poly6=rng.choice([0, 0, 0, 1]))
    if kind == "edges":
        return dict(kind=kind, scene="tank", particles=n, precision=prec, edges=_log_int(rng, 500, 400000))
    return dict(kind=kind, scene="tank", particles=n, queries=_log_int(rng, 500, 600000))


def _frame_sizes(case):
    """Particles of each frame of a batch: uneven, the largest neither first nor last."""
    for k in range(case["frames"]):
        t = ((2 * k + 1) % case["frames"]) / max(case["frames"] - 1, 1)
        yield int(case["smallest"] * (case["largest"] / case["smallest"]) ** t)


# ---- inputs --------------------------------------------------------------------------------
def _points(case, x, r, g):
    """Query points around the particles: a particle's position moved by up to 3 r per axis, in
    random order or in the order of the particles."""
    pick = torch.randint(0, len(x), (case["points"],), generator=g, device="cuda")
    if case["order"] == "scan":
        pick = pick.sort().values
    return (x[pick].double() + _uniform(g, (case["points"], 3), -3 * r, 3 * r)).float()


def _edge_points(case, x, r, g, want):
    """Ends of axis-parallel dual edges of length r or 2 r near the tank's free surface, and a key that
    orders them tile by tile (as an extraction in space-filling order hands them over)."""
    top = x[x[:, 2] > 0.15].double()
    pick = torch.randint(0, len(top), (want,), generator=g, device="cuda")
    a = top[pick] + _uniform(g, (want, 3), -r, r)
    step = torch.where(_uniform(g, (want,)) < 0.5, 1.0, 2.0) * r
    axis = torch.randint(0, 3, (want,), generator=g, device="cuda")
    sign = torch.where(_uniform(g, (want,)) < 0.5, 1.0, -1.0)
    b = a.clone()
    b[torch.arange(want, device="cuda"), axis] += sign * step
    tile = torch.floor(a / (4 * r)).long()
    return a.float(), b.float(), (tile[:, 2] * 4096 + tile[:, 1]) * 4096 + tile[:, 0]


def _context(case, x, r):
    ctx = capi.Context(0)
    ctx.set_params(r, precision=PREC[case.get("precision", "fp32")], use_ani=case.get("ani", 1),
                   use_poly6=case.get("poly6", 0), qef_mode=QEF[case.get("qef", "off")],
                   depth_max_override=case.get("depth", 0))
    return ctx


def _on_device(ctx, x):
    torch.cuda.synchronize()
    ctx.upload(None, device_ptr=x.data_ptr(), n=len(x))


class _Mesh:
    """Buffers that a program's frame loop keeps for the mesh: room for more than the frame's
    vertices and triangles, so that every frame of the sequence fits."""

    def __init__(self, case):
        usual = case.get("ani", 1) and not case.get("poly6", 0)
        cap = int((1.6 if usual else 6.0) * _surface_points(case)) + 30000
        self.verts = np.full((cap, 3), 0.0)
        self.tris = np.full((cap * 9 // 4, 3), 0, np.int32)

    def hold(self, nv, nt):
        if nv > len(self.verts) or nt > len(self.tris):
            raise RuntimeError("mesh of %d vertices and %d triangles: more than the buffers hold" % (nv, nt))


def _ptr(a):
    return a.ctypes.data_as(C.c_void_p)


def prepare(case, seed):
    s = dict(kind=case["kind"], case=case)
    if case["kind"] == "batch":
        s["frames"], radii, s["mesh"] = [], [], []
        for k, n in enumerate(_frame_sizes(case)):
            x, r = _tank(_gen(seed * 1000 + k), case, n)
            s["frames"].append(x.float().cpu().numpy())
            s["mesh"].append(_Mesh(dict(scene="tank", particles=n)))
            radii.append(r)
        m = case["frames"]
        s["xyz"] = (C.c_void_p * m)(*[f.ctypes.data for f in s["frames"]])
        s["n"] = (C.c_int64 * m)(*[len(f) for f in s["frames"]])
        s["radii"] = (C.c_float * m)(*radii)
        s["ctx"] = _context(case, None, radii[0])
        return s
    x, r, g = _particles(case, seed)
    s["ctx"] = ctx = _context(case, x, r)
    if case["kind"] == "frame":
        s["x"] = x.cpu().numpy() if case["input"] == "host" else x
        s["mesh"] = _Mesh(case)
    elif case["kind"] == "points":
        s["q"] = _points(case, x, r, g).cpu().numpy()
        s["x"] = x
        if not case["fresh"]:
            _on_device(ctx, x)
            ctx.anisotropy()
    elif case["kind"] == "lattice":
        _on_device(ctx, x)
        ctx.anisotropy()
        s["values"] = np.full(_lattice_room(case), 0, np.float32)
    elif case["kind"] == "edges":
        _on_device(ctx, x)
        ctx.anisotropy()
        a, b, tile = _edge_points(case, x, r, g, 12 * case["edges"] + 20000)
        fa = torch.from_numpy(ctx.eval_points(a.cpu().numpy())).cuda()
        fb = torch.from_numpy(ctx.eval_points(b.cpu().numpy())).cuda()
        keep = torch.nonzero((fa > 0) != (fb > 0)).flatten()
        keep = keep[torch.arange(case["edges"], device="cuda") % len(keep)]
        keep = keep[tile[keep].sort(stable=True).indices]
        ends = torch.stack([torch.cat([a.double(), fa[:, None]], 1), torch.cat([b.double(), fb[:, None]], 1)], 1)
        s["ends"] = ends[keep].contiguous().cpu().numpy()
    else:
        _on_device(ctx, x)
        ctx.hashgrid_build()
        pick = torch.randint(0, len(x), (case["queries"],), generator=g, device="cuda").sort().values
        s["q"] = x[pick].contiguous()
        s["offsets"] = torch.empty(case["queries"] + 1, dtype=torch.int64, device="cuda")
        s["ids"] = torch.zeros(300 * case["queries"] + 100000, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    return s


def _check(ctx, rc):
    if rc != 0:
        raise capi.PisurfError("%d: %s" % (rc, ctx.L.pisurf_last_error(ctx.h).decode()))


# ---- one pass ------------------------------------------------------------------------------
def run(s):
    ctx, case = s["ctx"], s["case"]
    if s["kind"] == "frame":
        if case["input"] == "host":
            ctx.upload(s["x"])
        else:
            ctx.upload(None, device_ptr=s["x"].data_ptr(), n=len(s["x"]))
        info = ctx.run_frame()
        st = ctx.stats()
        mesh = s["mesh"]
        mesh.hold(st["n_verts"], st["n_tris"])
        _check(ctx, ctx.L.pisurf_mesh_download(ctx.h, _ptr(mesh.verts), _ptr(mesh.tris)))
        return dict(verts=mesh.verts, tris=mesh.tris, n_verts=st["n_verts"], n_tris=st["n_tris"], nodes=info["n_nodes"])
    if s["kind"] == "batch":
        counts = [None] * case["frames"]

        def on_mesh(user, k, tree, verts, nv, tris, nt):
            mesh = s["mesh"][k]
            if nv <= len(mesh.verts) and nt <= len(mesh.tris):
                C.memmove(mesh.verts.ctypes.data, verts, 24 * nv)
                C.memmove(mesh.tris.ctypes.data, tris, 12 * nt)
                counts[k] = (nv, nt)

        _check(ctx, ctx.L.pisurf_run_frames(ctx.h, case["frames"], s["xyz"], s["n"], s["radii"], 0,
                                            capi.MESH_CB(on_mesh), None, None))
        return dict(verts=[m.verts for m in s["mesh"]], tris=[m.tris for m in s["mesh"]], counts=counts)
    if s["kind"] == "points":
        if case["fresh"]:
            ctx.upload(None, device_ptr=s["x"].data_ptr(), n=len(s["x"]))
            ctx.anisotropy()
        if case["grad"]:
            f, grad = ctx.eval_points(s["q"], grad=True)
            return dict(f=f, grad=grad)
        return dict(f=ctx.eval_points(s["q"]))
    if s["kind"] == "lattice":
        dims, box, spacing = (C.c_int32 * 3)(), (C.c_float * 6)(), C.c_float()
        _check(ctx, ctx.L.pisurf_uniform_grid(ctx.h, dims, box, C.byref(spacing), None))
        if dims[0] * dims[1] * dims[2] > len(s["values"]):
            raise RuntimeError("lattice of %s points: more than the buffer holds" % (list(dims),))
        _check(ctx, ctx.L.pisurf_uniform_grid(ctx.h, None, None, None, _ptr(s["values"])))
        return dict(values=s["values"], dims=list(dims), box=list(box), spacing=spacing.value)
    if s["kind"] == "edges":
        verts, evals = ctx.bisect_edges(s["ends"])
        return dict(verts=verts, evals=evals)
    total = C.c_int64()
    q, offsets, ids = s["q"], s["offsets"], s["ids"]
    _check(ctx, ctx.L.pisurf_neighbors_noalloc(ctx.h, C.c_void_p(q.data_ptr()), C.c_int64(len(q)),
                                               C.c_void_p(offsets.data_ptr()), C.c_void_p(ids.data_ptr()),
                                               C.c_int64(len(ids)), C.byref(total)))
    return dict(offsets=offsets, ids=ids, total=total.value)


# ---- the work of a pass --------------------------------------------------------------------
# In the inside of a lattice of spacing 2 r about 33 particles lie within the kernel's 4 r. One
# neighbour's share: about 20 operations for the mean, 40 for the covariance, 35 for the field and
# 10 more for the gradient.
NEAR = 33


def _surface_points(case):
    """Lattice points of spacing r on the fluid's surface, about."""
    if case["scene"] == "dam":
        return 2.6e4
    if case["scene"] == "tank":
        r = (0.0125 / case["particles"]) ** (1.0 / 3.0)
        return 1.6 / r ** 2
    if case["scene"] == "crown":
        return (0.72 + 2.4 * 0.002 * case["layers"] + 1.2) / 1e-6
    return (0.5 + 2.0 * 0.001 * case["layers"] + 0.04) / 2.5e-7 + 2e6


def _lattice_room(case):
    """Points of the dense lattice at most: the tank's box with its spray, spacing r."""
    r = (0.0125 / case["particles"]) ** (1.0 / 3.0)
    return int((1.2 / r + 40) * (0.7 / r + 40) * (0.42 / r + 40))


def _frame_work(case):
    n, surf = _count(case), _surface_points(case)
    # a vertex (24 B) and two triangles (12 B each) per surface lattice point; about 12 field values
    # for each of them, and for each particle its mean, its covariance and its normal
    return dict(bytes=12 * n + 48 * surf, flops=NEAR * (n * (20 + 40 + 45) + 12 * surf * 35))


def work(case):
    if case["kind"] == "frame":
        return _frame_work(case)
    if case["kind"] == "batch":
        w = dict(bytes=0, flops=0)
        for n in _frame_sizes(case):
            one = _frame_work(dict(scene="tank", particles=n))
            w = {key: w[key] + one[key] for key in w}
        return w
    n = _count(case)
    if case["kind"] == "points":
        m = case["points"]
        w = dict(bytes=m * (12 + 8 + 24 * case["grad"]), flops=NEAR * m * (35 + 10 * case["grad"]))
        # the particle records around the points are read once
        w["bytes"] += 52 * min(n, NEAR * m) if not case["fresh"] else 12 * n
        w["flops"] += NEAR * n * 60 if case["fresh"] else 0
        return w
    if case["kind"] == "lattice":
        m = 0.2 * 0.5 * 1.3 / (0.0125 / case["particles"])  # box volume over r^3
        return dict(bytes=4 * m + 52 * n, flops=NEAR * 0.5 * m * 35)
    if case["kind"] == "edges":
        return dict(bytes=case["edges"] * (64 + 24 + 4), flops=NEAR * case["edges"] * 2 * 35)
    return dict(bytes=case["queries"] * (12 + 8 + 4 * 190), flops=case["queries"] * 50)


# ---- 64-bit values -------------------------------------------------------------------------
class _Field:
    """Anisotropic B-spline field of a particle set in double (Evaluator of the reference): particles
    binned by their float positions, sums over the 27 cells around a point."""

    def __init__(self, x, r):
        f4 = np.float32
        self.r = f4(r)
        cell = f4(self.r * f4(4))
        lo, hi = x.min(0).values.cpu().numpy(), x.max(0).values.cpu().numpy()
        length = np.ceil((hi - lo) / cell).astype(f4) * cell
        centre = (lo + hi) / f4(2)
        self.b0 = (centre - length / f4(2)).astype(f4)
        b1 = (centre + length / f4(2)).astype(f4)
        self.n = [max(int(math.ceil(v)), 1) for v in (b1 - self.b0) / cell]
        self.cell = cell
        c = self._cells(x)
        inside = ((c >= 0) & (c < torch.tensor(self.n, device=x.device))).all(1)
        key = torch.where(inside, (c[:, 2] * self.n[1] + c[:, 1]) * self.n[0] + c[:, 0], -1)
        if not bool(inside.all()):
            raise ValueError("particles outside the grid")
        key, order = key.sort(stable=True)
        self.x = x[order].double()
        self.off = torch.searchsorted(key, torch.arange(self.n[0] * self.n[1] * self.n[2] + 1, device=x.device))
        h = float(f4(self.r * f4(2)))
        self.h2, self.sigma = h * h, 1.0 / h ** 6
        q = float(f4(0.01))
        self.iso = self.sigma * (1 - 1.5 * q ** 2 + 0.75 * q ** 3)
        self._anisotropy(x[order])

    def _cells(self, p):
        b0 = torch.from_numpy(self.b0).to(p.device)
        v = (p - b0) / torch.tensor(self.cell, device=p.device)
        return v.clamp(-8, 1 << 20).to(torch.int64)  # truncation toward zero

    def _pairs(self, p, visit):
        """visit(i, j) for index tensors of points i and candidates j, each pair once."""
        c = self._cells(p)
        for d in range(27):
            e = c + torch.tensor([d % 3 - 1, (d // 3) % 3 - 1, d // 9 - 1], device=p.device)
            ok = ((e >= 0) & (e < torch.tensor(self.n, device=p.device))).all(1)
            i = torch.nonzero(ok).flatten()
            k = (e[i, 2] * self.n[1] + e[i, 1]) * self.n[0] + e[i, 0]
            j, end = self.off[k], self.off[k + 1]
            while True:
                more = j < end
                i, j, end = i[more], j[more], end[more]
                if not len(i):
                    break
                visit(i, j)
                j = j + 1

    def _anisotropy(self, xf):
        n, x = len(self.x), self.x
        nI = float(np.float32(self.r * np.float32(4)))
        nI2 = float(np.float32(nI) * np.float32(nI))

        def w_of(d):
            return torch.where(d < nI, torch.where(d < nI / 2, 1 - 6 * d * d * (nI - d) / nI ** 3,
                                                   2 * (nI - d) ** 3 / nI ** 3), torch.zeros_like(d))

        acc = torch.zeros(n, 5, device=x.device, dtype=torch.float64)

        def mean(i, j):
            d = x[j] - x[i]
            d2 = (d * d).sum(1)
            w = torch.where((d2 < nI2) & (i != j), w_of(d2.sqrt()), torch.zeros_like(d2))
            acc[i] += torch.cat([x[j] * w[:, None], w[:, None], torch.ones_like(w)[:, None]], 1)

        self._pairs(xf, mean)
        b = float(np.float32(0.9))
        ok = (acc[:, 4] > 2) & (acc[:, 3] > 0)
        self.xm = torch.where(ok[:, None], x * float(np.float32(1) - np.float32(0.9)) + acc[:, :3] / acc[:, 3:4] * b, x)
        xm = self.xm
        cov = torch.zeros(n, 7, device=x.device, dtype=torch.float64)

        def second(i, j):
            d = xm[j] - xm[i]
            d2 = (d * d).sum(1)
            w = torch.where(d2 < nI2, w_of(d2.sqrt()), torch.zeros_like(d2))
            a, bb, c = d[:, 0], d[:, 1], d[:, 2]
            cov[i] += torch.stack([a * a, a * bb, a * c, bb * bb, bb * c, c * c, torch.ones_like(w)], 1) * w[:, None]

        self._pairs(xf, second)
        m = cov[:, :6].clone()
        for k in (0, 3, 5):
            m[:, k] += self.h2
        m /= cov[:, 6:7]
        self.G, self.det = self._g(m)

    @staticmethod
    def _g(m):
        """G and its determinant from the covariances (Jacobi eigenvalues, |l| clamped at max / 4)."""
        A = torch.stack([m[:, 0], m[:, 1], m[:, 2], m[:, 1], m[:, 3], m[:, 4], m[:, 2], m[:, 4], m[:, 5]], 1).view(-1, 3, 3)
        Q = torch.eye(3, device=m.device, dtype=torch.float64).repeat(len(m), 1, 1)
        for _ in range(8):
            for p, q in ((0, 1), (0, 2), (1, 2)):
                apq = A[:, p, q]
                tau = (A[:, q, q] - A[:, p, p]) / (2 * torch.where(apq == 0, torch.ones_like(apq), apq))
                t = torch.where(tau >= 0, 1.0, -1.0) / (tau.abs() + (1 + tau * tau).sqrt())
                t = torch.where(apq == 0, torch.zeros_like(t), t)
                c = 1 / (1 + t * t).sqrt()
                s = t * c
                J = torch.eye(3, device=m.device, dtype=torch.float64).repeat(len(m), 1, 1)
                J[:, p, p], J[:, q, q], J[:, p, q], J[:, q, p] = c, c, s, -s
                A = (J.transpose(1, 2)[:, :, :, None] * A[:, None, :, :]).sum(2)
                A = (A[:, :, :, None] * J[:, None, :, :]).sum(2)
                Q = (Q[:, :, :, None] * J[:, None, :, :]).sum(2)
        w = torch.stack([A[:, 0, 0], A[:, 1, 1], A[:, 2, 2]], 1).abs()
        w = torch.maximum(w, w.max(1, keepdim=True).values / 4)
        s = w.prod(1) ** (1.0 / 3.0)
        G = (Q[:, :, None, :] * (s[:, None] / w)[:, None, None, :] * Q[:, None, :, :]).sum(3)
        return G, (s ** 3) / w.prod(1)

    def value(self, q, grad=False):
        """Field (and the gradient of its poly6 form) at float or double points q."""
        p = q.double()
        f = torch.zeros(len(p), 4 if grad else 1, device=p.device, dtype=torch.float64)

        def add(i, j):
            d = p[i] - self.xm[j]
            g = (self.G[j] * d[:, None, :]).sum(2)
            n2 = (g * g).sum(1)
            u2 = n2 / self.h2
            u = u2.sqrt()
            k = torch.where(u2 < 4, torch.where(u <= 1, 1 - 1.5 * u2 + 0.75 * u2 * u, 0.25 * (2 - u) ** 3),
                            torch.zeros_like(u))
            v = (self.det[j] * k)[:, None]
            if grad:
                t = torch.where(n2 > self.h2, torch.zeros_like(n2), self.h2 - n2)
                v = torch.cat([v, (-6 * self.det[j] * t * t)[:, None] * g], 1)
            f[i] += v

        self._pairs(q.float(), add)
        out = self.iso - self.sigma * f[:, 0]
        return (out, self.sigma * f[:, 1:]) if grad else out


def exact(case, seed):
    # A mesh follows a tree of decisions and has no value of its own in 64 bits; neighbour lists are
    # whole numbers. The double field here is the default kernel's.
    if case["kind"] not in ("points", "lattice", "edges") or case.get("poly6", 0) or not case.get("ani", 1):
        return None
    if case["kind"] == "edges":
        return None  # which end a midpoint replaces, and the snap to an end, are decisions too
    x, r, g = _particles(case, seed)
    if case["kind"] == "points":
        q = _points(case, x, r, g)
        field = _Field(x, r)
        if case["grad"]:
            f, grad = field.value(q, True)
            return dict(f=f, grad=grad)
        return dict(f=field.value(q))
    # the lattice of UniformGrid: the particles' box, each axis grown to whole radii and 4 r more
    field = _Field(x, r)
    f4 = np.float32
    lo, hi = x.min(0).values.cpu().numpy(), x.max(0).values.cpu().numpy()
    axes = []
    for a in range(3):
        centre = f4((lo[a] + hi[a]) / f4(2))
        length = f4(f4(np.ceil(f4(f4(hi[a] - lo[a]) / field.r)) * field.r) + f4(field.r * f4(4)))
        b0, b1 = f4(centre - length / f4(2)), f4(centre + length / f4(2))
        steps = int(f4(length / field.r))
        i = np.arange(steps + 1).astype(f4)
        axes.append((f4(steps) - i) / f4(steps) * b0 + i / f4(steps) * b1)
    X, Y, Z = (torch.from_numpy(v.astype(f4)).cuda() for v in axes)
    z, y, xx = torch.meshgrid(Z, Y, X, indexing="ij")
    pts = torch.stack([xx, y, z], -1).reshape(-1, 3)
    values = torch.cat([field.value(c) for c in pts.split(1 << 22)])
    room = torch.zeros(_lattice_room(case), dtype=torch.float64, device="cuda")
    room[:len(values)] = values
    return dict(values=room, dims=None, box=None, spacing=None)
