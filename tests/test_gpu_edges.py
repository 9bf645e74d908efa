"""The trace kernels, node quantisation, grouped build, domain lists and paged
images at the edges of their ranges, against the oracle: batch sizes around a
wave's share of a launch, meshes that are flat, far, vast, tiny or deep, domain
counts around a launch's group, images of a few pixels, meshes with and without
shared vertices in a partial cache, and contexts that change scene and size.

Hits use the oracle's arithmetic, so they are compared bit for bit with its
brute force over every triangle, which depends on no box; images within 1e-4
RMS and 1e-3, as everywhere."""
import math
import os

import numpy as np
import pytest

import orc
import scenes

pytestmark = pytest.mark.gpu

CAM = dict(pos=[1.5, 1.5, 4.5], lookat=[1.5, 1.5, 1.5], up=[0.0, 1.0, 0.0])
LIGHT = "light rect 0.5 3.4 0.5 2 0 0 0 0 2 4 4 4"


def _soup(rng, n, size=0.08):
    """n separate triangles in the unit cube."""
    c = rng.uniform(0.1, 0.9, (n, 1, 3))
    v = (c + rng.uniform(-size, size, (n, 3, 3))).reshape(-1, 3)
    return v, np.arange(3 * n).reshape(-1, 3)


def _sheet(rng, k, bump=0.1):
    """A k x k grid of shared vertices, 2 k^2 triangles."""
    y, x = np.mgrid[0:k + 1, 0:k + 1] / k
    v = np.stack([x, y, 0.5 + bump * rng.uniform(-1, 1, x.shape)], -1).reshape(-1, 3)
    i = (np.arange(k)[:, None] * (k + 1) + np.arange(k)).reshape(-1)
    f = np.concatenate([np.stack([i, i + 1, i + k + 1], -1), np.stack([i + 1, i + k + 2, i + k + 1], -1)])
    return v, f


def _rays_at(rng, verts, faces, n):
    """Rays towards points of the mesh, a third of them along an axis, and
    some that miss it."""
    v = np.asarray(verts, np.float32).astype(np.float64)
    tri = v[np.asarray(faces)[rng.integers(0, len(faces), n)]]
    w = rng.dirichlet([1.0, 1.0, 1.0], n)
    tgt = (tri * w[:, :, None]).sum(1)
    ext = np.max(v.max(0) - v.min(0))
    d = rng.normal(size=(n, 3))
    ax = np.arange(n) % 9
    d[ax < 3] = np.eye(3)[ax[ax < 3]]
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    org = tgt - d * (ext + 1.0) * rng.uniform(0.5, 2.0, (n, 1))
    miss = np.arange(n) % 11 == 0
    d[miss] = -d[miss]
    return org.astype(np.float32), d.astype(np.float32)


def _check(ctx, ref, dom, org, dirs, tfar=None):
    t, u, v, p = ctx.trace_rays(org, dirs, dom)
    rt, ru, rv, rp = ref.closest(dom, org, dirs, brute=True)
    assert np.array_equal(p, rp) and np.array_equal(t, rt), dom
    hit = rp >= 0
    assert np.array_equal(u[hit], ru[hit]) and np.array_equal(v[hit], rv[hit]), dom
    assert np.array_equal(ctx.trace_rays(org, dirs, dom, mode=1), hit), dom
    return int(hit.sum())


def _load(tmp_path, domains, cache=-1, **cfg):
    import spray_amd as sa
    path = scenes.write_scene(str(tmp_path), "s", domains, [LIGHT])
    ctx = sa.Context(sa.default_config(nthreads=8, **cfg))
    if cache >= 0:
        ctx.set_cache_size(cache)
    ctx.load_scene(path, str(tmp_path))
    return ctx, orc.Scene(path, str(tmp_path))


@pytest.mark.parametrize("n", [1, 3, 4, 5, 63, 64, 65, 255, 257, 16383, 16385, 65537])
def test_query_batch_sizes(tmp_path, n):
    rng = np.random.default_rng(n)
    v, f = _soup(rng, 700)
    ctx, ref = _load(tmp_path, [dict(verts=v, faces=f)])
    with ctx:
        org, dirs = _rays_at(rng, v, f, n)
        hits = _check(ctx, ref, 0, org, dirs)
    assert n < 63 or 0 < hits < n


def _shape(kind, rng):
    if kind in ("1", "2", "3"):
        return _soup(rng, int(kind), 0.4)
    v, f = _soup(rng, 600)
    if kind == "flat":
        v[:, 2] = 0.25
    elif kind == "thin":
        v = v * [1.0, 1e-6, 1.0]
    elif kind == "far":
        v = v + [9000.0, -7000.0, 8500.0]
    elif kind == "tiny":
        v = v * 1e-5
    elif kind == "huge":
        v = v * 1e12
    elif kind == "vast":  # one triangle that spans 1e25: axes whose step would exceed every limit
        v[:3] = [[-1e25, -1e25, 5e24], [1e25, -1e25, 5e24], [0.0, 1e25, 5e24]]
    elif kind == "degenerate":  # a third points, a third segments
        v[0::9] = v[1::9] = v[2::9]
        v[3::9] = v[4::9]
    elif kind == "coincident":
        v = np.tile(v[:6], (200, 1))
        f = np.arange(len(v)).reshape(-1, 3)
    elif kind == "deep":  # ever smaller copies around a corner: a chain of nodes
        c = [_soup(rng, 60)[0] * 2.0 ** -s for s in range(20)]
        v = np.concatenate(c)
        f = np.arange(len(v)).reshape(-1, 3)
    return v, f


@pytest.mark.parametrize("builder", [0, 1])
@pytest.mark.parametrize("kind", ["1", "2", "3", "flat", "thin", "far", "tiny", "huge", "vast", "degenerate",
                                  "coincident", "deep"])
def test_mesh_shapes(tmp_path, kind, builder):
    import spray_amd as sa
    rng = np.random.default_rng(5)
    v, f = _shape(kind, rng)
    path = scenes.write_scene(str(tmp_path), "s", [dict(verts=v, faces=f)], [])
    ref = orc.Scene(path, str(tmp_path))
    with sa.Context(sa.default_config(nthreads=8)) as ctx:
        ctx.set_bvh_builder(builder)
        ctx.load_scene(path, str(tmp_path))
        aim = slice(3, None) if kind == "vast" else slice(None)
        org, dirs = _rays_at(rng, v if kind != "vast" else np.where(np.abs(v) > 1e20, 0.5, v), f[aim], 3000)
        hits = _check(ctx, ref, 0, org, dirs)
        assert np.array_equal(ctx.normals(0), ref.mesh(0)[3])
    assert hits > 0 or kind in ("thin", "tiny", "degenerate")


@pytest.mark.parametrize("nd", [2, 16, 17, 33])
def test_grouped_build(tmp_path, nd):
    """Domains of 1 to 392 triangles in one build, whose launches take up to 16."""
    rng = np.random.default_rng(nd)
    doms = []
    for d in range(nd):
        v, f = _sheet(rng, 14) if d % 5 == 4 else _soup(rng, (1, 2, 3, 40)[d % 5], 0.3)
        doms.append(dict(verts=v + [d % 6, d // 6, 0.0], faces=f))
    ctx, ref = _load(tmp_path, doms)
    with ctx:
        for d, dom in enumerate(doms):
            org, dirs = _rays_at(rng, dom["verts"], dom["faces"], 400)
            _check(ctx, ref, d, org, dirs)
            assert np.array_equal(ctx.normals(d), ref.mesh(d)[3])


def _frame_ok(ctx, ref, **kw):
    img, st = ctx.trace_frame()
    rimg, rst = ref.render(nthreads=8, cam_pos=CAM["pos"], cam_lookat=CAM["lookat"], cam_up=CAM["up"], **kw)
    err = np.abs(img[..., :3] - rimg[..., :3])
    assert st["useful_rays"] == rst["useful_rays"] and st["final_hits"] == rst["final_hits"]
    assert math.sqrt(float((err ** 2).mean())) <= 1e-4 and float(err.max()) <= 1e-3


def _cfg(**kw):
    import spray_amd as sa
    return sa.default_config(has_camera=1, camera_pos=CAM["pos"], camera_lookat=CAM["lookat"],
                             camera_up=CAM["up"], nthreads=8, **kw)


@pytest.fixture(scope="module")
def lattices(tmp_path_factory):
    import spray_amd as sa
    d = str(tmp_path_factory.mktemp("edges"))
    sa.scenegen_write(d, "g27", 3, 3, 3, 20, rgb=0xB3B3B3, extra_lines=LIGHT)
    sa.scenegen_write(d, "g2", 2, 1, 1, 6, rgb=0xB3B3B3, extra_lines=LIGHT)
    return d, {k: orc.Scene(os.path.join(d, k + ".spray"), d) for k in ("g27", "g2")}


@pytest.mark.parametrize("schedule", [0, 1])
@pytest.mark.parametrize("size", [(1, 1), (3, 2), (17, 5), (64, 63)])
def test_small_frames(lattices, size, schedule):
    import spray_amd as sa
    d, ref = lattices
    kw = dict(image_w=size[0], image_h=size[1], pixel_samples=1, ao_mode=0, ao_samples=1, bounces=4, rr_start=3)
    with sa.Context(_cfg(schedule=schedule, **kw)) as ctx:
        ctx.load_scene(os.path.join(d, "g27.spray"), d)
        _frame_ok(ctx, ref["g27"], **kw)


@pytest.mark.parametrize("schedule", [0, 1])
@pytest.mark.parametrize("ao,bounces", [(1, 1), (1, 3), (0, 1), (0, 2), (0, 4), (0, 5), (0, 9)])
def test_passes_of_a_window(lattices, ao, bounces, schedule):
    """Paths that end within, at and beyond a window of four depths."""
    import spray_amd as sa
    d, ref = lattices
    kw = dict(image_w=24, image_h=20, pixel_samples=2, ao_mode=ao, ao_samples=2, bounces=bounces, rr_start=6,
              ao_max_dist=0.5)
    with sa.Context(_cfg(schedule=schedule, **kw)) as ctx:
        ctx.load_scene(os.path.join(d, "g27.spray"), d)
        _frame_ok(ctx, ref["g27"], **kw)


def test_context_changes_scene_and_size(lattices):
    """One context's memory serves other scenes and sizes: larger, smaller and
    larger again, each frame as the oracle's."""
    import spray_amd as sa
    d, ref = lattices
    first = True
    for scene, w, h, schedule in (("g2", 8, 8, 1), ("g27", 96, 64, 1), ("g2", 96, 64, 0), ("g2", 5, 3, 1),
                                  ("g27", 130, 40, 1), ("g27", 16, 16, 0)):
        kw = dict(image_w=w, image_h=h, pixel_samples=2, ao_mode=0, ao_samples=1, bounces=3, rr_start=3)
        cfg = _cfg(schedule=schedule, **kw)
        if first:
            ctx = sa.Context(cfg)
            first = False
        else:
            ctx.set_config(cfg)
        ctx.load_scene(os.path.join(d, scene + ".spray"), d)
        _frame_ok(ctx, ref[scene], **kw)
        _frame_ok(ctx, ref[scene], **kw)
    ctx.close()


@pytest.mark.parametrize("cache", [1, 2, 5])
def test_paged_images_of_both_forms(tmp_path, cache):
    """Domains with shared vertices (their mesh crosses the host link) and
    without (their finished arrays do), one of them of a single triangle:
    hits and normals while domains are loaded and evicted."""
    rng = np.random.default_rng(9)
    doms = []
    for d in range(6):
        v, f = _sheet(rng, 12) if d % 2 else _soup(rng, 1 if d == 4 else 90)
        doms.append(dict(verts=v + [d, 0.0, 0.0], faces=f))
    ctx, ref = _load(tmp_path, doms, cache=cache)
    with ctx:
        for turn in range(2):
            for d in (0, 5, 1, 4, 2, 3):
                org, dirs = _rays_at(rng, doms[d]["verts"], doms[d]["faces"], 300)
                assert _check(ctx, ref, d, org, dirs) > 0
                assert np.array_equal(ctx.normals(d), ref.mesh(d)[3])
