"""Performance cases: the work a program does with this framework.

Every case goes through the public entry points (spray_amd.Context, and the
C ABI where the Python class has no method of its own) on synthetic scenes of
the kinds the benchmark and the tests use: lattices of marching-cubes
isosurface domains, the same number of cells in every domain ("even") or
log-uniform triangle budgets ("uneven"), and a single-domain height field for
the ray query interface.

Kinds of case:
  frame   one frame of a loaded scene: ambient occlusion ("ao") or path
          tracing ("pt"), with the plain, batched or learned schedule, the
          whole scene in HBM or a domain cache smaller than the scene
  insitu  the in-situ step: the scene remeshed at a new field phase, then one
          frame of it
  load    a run's start: PLY files and a .spray file loaded, then one frame
  rays    closest-hit or any-hit queries of ray batches on one domain, in
          device memory

A frame's outputs are its image and the two ray counts that every schedule
shares; a query's outputs are all its per-ray results.
"""
import ctypes
import math
import os
import random
import tempfile

import numpy as np
import torch

import spray_amd as sa

SCHEDULES = {"plain": 0, "batched": 1, "learned": 2}

# samples of one predictor batch, and (ray, domain, hit) samples logged for it
TRAIN_BATCH = 4096
TRAIN_SAMPLES = 1 << 19


def _frame(name, grid, mesh, image, spp, mode, schedule, bounces, kind="frame", res=0, tris=0,
           cache=0, shininess=0.0):
    nx, ny, nz = grid
    return dict(name=name, kind=kind, nx=nx, ny=ny, nz=nz, mesh=mesh, res=res, tris=tris, w=image[0],
                h=image[1], spp=spp, mode=mode, ao_samples=8 if mode == "ao" else 1, bounces=bounces,
                schedule=schedule, cache=cache, shininess=shininess)


def listed():
    return [
        # an interactive preview: a few domains, a thumbnail, one sample per pixel
        _frame("preview_ao", (2, 2, 2), "even", (96, 72), 1, "ao", "batched", 1, res=24),
        # the benchmark's ambient-occlusion frame on 64 domains
        _frame("ao_64dom", (4, 4, 4), "even", (512, 512), 1, "ao", "batched", 1, res=64),
        # the benchmark's 64-domain path-traced frame
        _frame("pt_64dom", (4, 4, 4), "even", (1024, 1024), 8, "pt", "batched", 5, res=64),
        # a production frame of the 256-domain scene with log-uniform domain
        # sizes (half the benchmark's triangles and samples, odd image size)
        _frame("pt_256dom", (8, 8, 4), "uneven", (1279, 719), 8, "pt", "batched", 6, tris=60_000_000),
        # the same kind of scene with the predictor ordering the visits
        _frame("pt_learned", (8, 8, 4), "uneven", (960, 540), 4, "pt", "learned", 6, tris=16_000_000),
        # the default schedule (reference order: one launch per scheduled domain)
        _frame("pt_plain", (3, 3, 3), "even", (256, 192), 2, "pt", "plain", 4, res=40),
        # out of core: a quarter of the domains cached in HBM, the rest paged in
        _frame("pt_paged", (4, 4, 3), "even", (400, 300), 4, "pt", "batched", 3, res=48, cache=12),
        # in situ: every domain remeshed, then a preview-quality frame
        _frame("insitu_step", (8, 4, 4), "even", (640, 360), 1, "pt", "batched", 8, kind="insitu", res=72),
        # start of a run: 27 binary PLY files read and built, first frame
        _frame("load_first_frame", (3, 3, 3), "even", (320, 240), 1, "ao", "batched", 1, kind="load",
               res=56),
        # ray queries on one domain: a large closest-hit batch, a large
        # any-hit (visibility) batch and a small closest-hit one
        dict(name="rays_closest", kind="rays", cells=512, n=3_000_000, any=False),
        dict(name="rays_visibility", kind="rays", cells=300, n=1_000_001, any=True),
        dict(name="rays_small", kind="rays", cells=48, n=1500, any=False),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "frame", "rays", "rays", "insitu", "load"])
    if kind == "rays":
        return dict(kind="rays", cells=_log(rng, 40, 500), n=_log(rng, 1000, 3_000_000),
                    any=rng.random() < 0.4)
    if kind == "frame":
        schedule = rng.choice(["batched", "batched", "batched", "learned", "plain", "paged"])
    else:
        schedule = "batched"
    small = kind != "frame" or schedule in ("plain", "paged")
    grid = [_log(rng, 2, 3 if schedule == "plain" else 4 if small else 8) for _ in range(3)]
    uneven = kind == "frame" and schedule in ("batched", "learned") and rng.random() < 0.5
    res, tris = 0, 0
    if uneven:
        tris = _log(rng, 200_000, 40_000_000)
    else:
        res = _log(rng, 16, 48 if small else 64)
    mode = rng.choice(["ao", "pt", "pt"])
    bounces = 1 if mode == "ao" else rng.randint(2, 4 if small and kind == "frame" else 8)
    most = 300_000 if small else 4_000_000
    w = _log(rng, 64, 640 if small else 1280)
    h = max(40, int(w * rng.uniform(0.5, 1.0)))
    spp = rng.choice([1, 1, 2, 4, 8]) if mode == "pt" else rng.choice([1, 1, 2])
    spp = max(1, min(spp, most // (w * h)))
    cache = max(2, grid[0] * grid[1] * grid[2] // 3) if schedule == "paged" else 0
    c = _frame("", tuple(grid), "uneven" if uneven else "even", (w, h), spp, mode,
               "batched" if schedule == "paged" else schedule, bounces, kind=kind, res=res, tris=tris,
               cache=cache, shininess=rng.choice([0.0, 0.0, 0.0, 20.0]))
    del c["name"]
    return c


# ---------------------------------------------------------------------------
def _lights(case):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if case["mode"] == "ao":
        return f"light point {nx / 2} {ny + 2} {nz / 2} 1 1 1"
    e1, e2 = max(0.5, nx - 1.0), max(0.5, nz - 1.0)
    return f"light rect 0.5 {ny + 0.5} 0.5 {e1} 0 0 0 0 {e2} 4 4 4"


def _config(case, rng):
    """Render settings and the camera: the scene's centre from +z at about half
    its diagonal (a little moved from seed to seed)."""
    ext = (case["nx"], case["ny"], case["nz"])
    diag = math.sqrt(sum(e * e for e in ext))
    look = [0.5 * e for e in ext]
    pos = [look[0] + rng.uniform(-0.2, 0.2), look[1] + rng.uniform(-0.2, 0.2),
           look[2] + 0.5 * diag * rng.uniform(1.0, 1.05)]
    pt = case["mode"] == "pt"
    kw = dict(image_w=case["w"], image_h=case["h"], pixel_samples=case["spp"], ao_mode=0 if pt else 1,
              ao_samples=case["ao_samples"], bounces=case["bounces"],
              ao_max_dist=math.inf if pt else 0.5, rr_start=3 if pt else 0, has_camera=1,
              camera_pos=pos, camera_lookat=look, camera_up=[0.0, 1.0, 0.0],
              schedule=SCHEDULES[case["schedule"]])
    if case["shininess"] > 0:
        kw.update(ks=[0.3, 0.3, 0.3], shininess=case["shininess"])
    return sa.default_config(nthreads=8, **kw)


def _scene(case, rng):
    """Scene generator arguments: the field's frequencies and phase move with the seed."""
    g = dict(nx=case["nx"], ny=case["ny"], nz=case["nz"], res=case["res"], a=rng.uniform(5.7, 6.3),
             b=rng.uniform(16.0, 18.0), phase=rng.uniform(0.0, 0.5),
             rgb=0xFFFFFF if case["mode"] == "ao" else 0xB3B3B3, extra_lines=_lights(case))
    if case["mesh"] == "uneven":
        g.update(per_domain_random=True, seed=rng.randrange(1 << 30), tri_total=float(case["tris"]))
    return g


class _State:
    """A context and the folder of its scene files, given back together."""

    def __init__(self, case):
        self.case = case
        self.ctx = None
        self.dir = None

    def __del__(self):
        if self.ctx is not None:
            self.ctx.close()
        if self.dir is not None:
            self.dir.cleanup()


def _prepare_frame(case, seed):
    rng = random.Random(seed)
    s = _State(case)
    cfg = _config(case, rng)
    gen = _scene(case, rng)
    s.phase = gen["phase"]
    s.ctx = sa.Context(cfg)
    if case["kind"] == "load" or case["cache"]:
        s.dir = tempfile.TemporaryDirectory(prefix="spray_perf_")
        sa.scenegen_write(s.dir.name, "scene", **gen)
        s.path = os.path.join(s.dir.name, "scene.spray")
    if case["kind"] == "load":
        return s
    if case["cache"]:
        s.ctx.set_cache_size(case["cache"])
        s.ctx.load_scene(s.path, s.dir.name)
    else:
        s.ctx.scenegen_load("scene", **gen)
    if case["schedule"] == "learned":  # the predictor learns from a batched frame's visits
        s.ctx.set_schedule(SCHEDULES["batched"])
        s.ctx.predictor_log(True, TRAIN_SAMPLES)
        s.ctx.trace_frame(want_image=False)
        s.ctx.predictor_log(False)
        s.ctx.predictor_train(1, TRAIN_BATCH, 2e-3)
        s.ctx.set_schedule(SCHEDULES["learned"])
    return s


def _height_field(cells, seed):
    """A wavy square sheet over [0, 1]^2 of 2 * cells^2 triangles: vertices, faces."""
    r = np.random.RandomState(seed % (1 << 31))
    f, p = r.uniform(5.0, 25.0, 6), r.uniform(0.0, 6.28, 6)
    g = np.linspace(0.0, 1.0, cells + 1)
    x, y = np.meshgrid(g, g, indexing="ij")
    z = 0.5 + 0.10 * np.sin(f[0] * x + p[0]) * np.sin(f[1] * y + p[1]) + \
        0.06 * np.sin(f[2] * x + f[3] * y + p[2]) + 0.02 * np.sin(3 * f[4] * x + p[4]) * np.sin(3 * f[5] * y)
    v = np.stack([x, y, z], -1).reshape(-1, 3).astype(np.float32)
    i = (np.arange(cells)[:, None] * (cells + 1) + np.arange(cells)[None, :]).reshape(-1)
    a, b, c, d = i, i + cells + 1, i + cells + 2, i + 1
    faces = np.concatenate([np.stack([a, b, c], 1), np.stack([a, c, d], 1)]).astype(np.int32)
    return v, faces


def _write_domain(directory, v, faces):
    with open(os.path.join(directory, "sheet.ply"), "wb") as fp:
        fp.write(("ply\nformat binary_little_endian 1.0\n"
                  f"element vertex {len(v)}\nproperty float x\nproperty float y\nproperty float z\n"
                  f"element face {len(faces)}\nproperty list uchar int vertex_indices\nend_header\n").encode())
        fp.write(v.astype("<f4").tobytes())
        rec = np.zeros(len(faces), dtype=[("n", "u1"), ("i", "<i4", 3)])
        rec["n"] = 3
        rec["i"] = faces
        fp.write(rec.tobytes())
    lo, hi = v.min(0), v.max(0)
    path = os.path.join(directory, "sheet.spray")
    with open(path, "w") as fp:
        fp.write("light point 0.5 0.5 3 1 1 1\ndomain\nfile sheet.ply\nmtl diffuse 1 1 1\nbound "
                 + " ".join(repr(float(t)) for t in list(lo) + list(hi))
                 + f"\nvertex {len(v)}\nface {len(faces)}\n")
    return path


def _rays(case, seed):
    """Rays around the sheet: origins in a box about it, directions everywhere,
    a quarter of them along one camera's view, half with a bounded length."""
    n = case["n"]
    g = torch.Generator(device="cuda").manual_seed(seed + 1)

    def uni(*shape):
        return torch.rand(*shape, generator=g, device="cuda", dtype=torch.float64)

    org = uni(n, 3) * 1.4 - 0.2
    z = 2.0 * uni(n) - 1.0
    phi = 2.0 * math.pi * uni(n)
    r = torch.sqrt(torch.clamp(1.0 - z * z, min=0.0))
    d = torch.stack([r * torch.cos(phi), r * torch.sin(phi), z], 1)
    m = n // 4  # one camera above the sheet, row by row
    side = max(1, int(math.sqrt(m)))
    k = torch.arange(m, device="cuda", dtype=torch.float64)
    at = torch.stack([torch.remainder(k, side) / side, torch.div(k, side, rounding_mode="floor") / side,
                      torch.full_like(k, 0.5)], 1)
    eye = torch.tensor([0.45, 0.4, 1.9], device="cuda", dtype=torch.float64)
    org[:m] = eye
    d[:m] = at - eye
    d = d / torch.linalg.norm(d, dim=1, keepdim=True)
    tfar = torch.full((n,), math.inf, device="cuda", dtype=torch.float32)
    half = n // 2
    tfar[half:] = (0.05 + 1.5 * uni(n - half)).to(torch.float32)
    return (org.to(torch.float32).contiguous(), d.to(torch.float32).contiguous(),
            torch.full((n,), 0.001, device="cuda", dtype=torch.float32), tfar)


def _prepare_rays(case, seed):
    s = _State(case)
    s.dir = tempfile.TemporaryDirectory(prefix="spray_perf_")
    path = _write_domain(s.dir.name, *_height_field(case["cells"], seed))
    s.ctx = sa.Context(sa.default_config(nthreads=8))
    s.ctx.load_scene(path, s.dir.name)
    s.org, s.dirs, s.tnear, s.tfar = _rays(case, seed)
    n = case["n"]
    s.t, s.u, s.v = (torch.empty(n, device="cuda", dtype=torch.float32) for _ in range(3))
    s.prim = torch.empty(n, device="cuda", dtype=torch.int32)
    torch.cuda.synchronize()
    return s


def prepare(case, seed):
    return _prepare_rays(case, seed) if case["kind"] == "rays" else _prepare_frame(case, seed)


# ---------------------------------------------------------------------------
def _fp(t):
    return ctypes.cast(t.data_ptr(), ctypes.POINTER(ctypes.c_float))


def run(state):
    case, ctx = state.case, state.ctx
    if case["kind"] == "rays":
        hit = not case["any"]
        rc = ctx.lib.spray_trace_rays_device(
            ctx.h, _fp(state.org), _fp(state.dirs), _fp(state.tnear), _fp(state.tfar), case["n"],
            _fp(state.t) if hit else None, _fp(state.u) if hit else None, _fp(state.v) if hit else None,
            ctypes.cast(state.prim.data_ptr(), ctypes.POINTER(ctypes.c_int)), 1 if case["any"] else 0, 0)
        if rc != 0:
            raise sa.SprayError(rc, ctx.lib.spray_last_error(ctx.h).decode())
        if hit:
            return {"t": state.t, "u": state.u, "v": state.v, "prim": state.prim}
        return {"prim": state.prim}
    if case["kind"] == "load":
        ctx.load_scene(state.path, state.dir.name)
    elif case["kind"] == "insitu":
        ctx.remesh(state.phase + 0.05)
    image, stats = ctx.trace_frame()
    return {"image": image, "useful_rays": stats["useful_rays"], "final_hits": stats["final_hits"]}


# ---------------------------------------------------------------------------
# What a pass cannot do without.  A ray's query costs at least the box tests
# of one path through a 4-wide hierarchy over its domain's triangles (24
# operations per box) and one triangle test (50); geometry is read once as
# vertices, indices and colours; a traced ray is written once and read once
# (origin, direction, weight, pixel: 40 bytes).
def _triangles(case):
    if case["mesh"] == "uneven":
        return float(case["tris"])
    # triangles per cells^2 of one domain of this field
    return 22.0 * case["res"] ** 2 * case["nx"] * case["ny"] * case["nz"]


def _query_flops(tris):
    return math.log(max(4.0, tris), 4) * 4 * 24 + 50


def work(case):
    if case["kind"] == "rays":
        tris = 2.0 * case["cells"] ** 2
        n = case["n"]
        return {"bytes": n * (32 + (4 if case["any"] else 16)) + tris * 18,
                "flops": n * _query_flops(tris)}
    tris = _triangles(case)
    domains = case["nx"] * case["ny"] * case["nz"]
    samples = case["w"] * case["h"] * case["spp"]
    # rays per sample: the eye ray and its occlusion rays, or about one bounce
    # ray and one light ray per vertex of the paths that Russian roulette keeps
    if case["mode"] == "ao":
        rays = samples * (1 + 0.5 * case["ao_samples"])
    else:
        rays = samples * (1 + 0.35 * min(case["bounces"], 5))
    n_bytes = rays * 80 + tris * 20 + case["w"] * case["h"] * 16
    flops = rays * _query_flops(tris / domains)
    if case["kind"] == "load":  # 7.5 file bytes per vertex and 13 per triangle, read once
        n_bytes += tris * 21
    if case["kind"] == "insitu":  # the field at every grid point; the mesh written once
        points = domains * (case["res"] + 1.0) ** 3
        n_bytes += tris * 20
        flops += points * 60
    return {"bytes": n_bytes, "flops": flops}


# ---------------------------------------------------------------------------
def exact(case, seed):
    """Ray queries against every triangle in float64 (Moeller-Trumbore); the
    frames' images have no closed value of this kind."""
    if case["kind"] != "rays" or case["any"]:
        return None
    tris = 2 * case["cells"] ** 2
    if tris * float(case["n"]) > 2e10:
        return None
    v, faces = _height_field(case["cells"], seed)
    org, dirs, tnear, tfar = (x.to(torch.float64) for x in _rays(case, seed))
    p = torch.from_numpy(v).cuda().to(torch.float64)
    f = torch.from_numpy(faces.astype(np.int64)).cuda()
    p0, e1, e2 = p[f[:, 0]], p[f[:, 1]] - p[f[:, 0]], p[f[:, 2]] - p[f[:, 0]]
    t_o, u_o, v_o = tfar.clone(), torch.zeros_like(tfar), torch.zeros_like(tfar)
    step = max(1, int(2e7 // tris))
    for b in range(0, case["n"], step):
        o, d = org[b:b + step, None, :], dirs[b:b + step, None, :]
        q = torch.linalg.cross(d, e2[None].expand(d.shape[0], -1, -1))
        det = (e1[None] * q).sum(-1)
        s = o - p0[None]
        r = torch.linalg.cross(s, e1[None].expand_as(s))
        inv = 1.0 / det
        u = (s * q).sum(-1) * inv
        w = (d * r).sum(-1) * inv
        t = (e2[None] * r).sum(-1) * inv
        ok = (u >= 0) & (w >= 0) & (u + w <= 1) & (t > tnear[b:b + step, None]) & (t < tfar[b:b + step, None])
        t = torch.where(ok, t, torch.full_like(t, math.inf))
        best, at = t.min(1)
        hit = torch.isfinite(best)
        rows = torch.arange(best.shape[0], device=best.device)
        t_o[b:b + step] = torch.where(hit, best, t_o[b:b + step])
        u_o[b:b + step] = torch.where(hit, u[rows, at], torch.zeros_like(best))
        v_o[b:b + step] = torch.where(hit, w[rows, at], torch.zeros_like(best))
    return {"t": t_o, "u": u_o, "v": v_o, "prim": None}
