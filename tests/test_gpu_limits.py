"""The trace kernels at the limits of a ray and of a tree, against the oracle's
brute force over every triangle (bit for bit, as the hits use its arithmetic)
and its frames: hits behind a ray's origin, trees so deep that a lane's stack
goes on in HBM, from host and from device arrays and in frames.  A ray may
visit as many nodes as its tree has, however many steps of its wave it waits
through: in the deep trees, of 200 nodes, those are many more."""
import math

import numpy as np
import pytest

import orc
import scenes
from test_gpu_edges import _load, _rays_at, _soup
from test_zz_no_alloc import _device_query

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,dist", [("soup", 1.0), ("soup", 1000.0), ("small", 30.0), ("small", 1000.0),
                                       ("flat", 1.0), ("flat", 30.0)])
def test_hits_behind_the_origin(tmp_path, kind, dist):
    """tnear below zero: what lies behind the origin is hit too, the farthest
    first, also where a box is thin against its distance."""
    rng = np.random.default_rng(3)
    v, f = _soup(rng, 3000, 0.002 if kind == "small" else 0.02)
    if kind == "flat":
        v[:, 2] = 0.25
    ctx, ref = _load(tmp_path, [dict(verts=v, faces=f)])
    org, dirs = _rays_at(rng, v, f, 20000)
    dirs = -dirs
    org = (org + dirs * np.float32(dist)).astype(np.float32)
    with ctx:
        for tnear, tfar in ((-math.inf, 0.0), (-math.inf, math.inf), (-2.0 * dist, -0.5)):
            t, u, w, p = ctx.trace_rays(org, dirs, 0, tnear=tnear, tfar=tfar)
            rt, ru, rw, rp = ref.closest(0, org, dirs, tnear=tnear, tfar=tfar, brute=True)
            assert np.array_equal(p, rp) and np.array_equal(t, rt), (tnear, tfar, int((p != rp).sum()))
            assert np.array_equal(ctx.trace_rays(org, dirs, 0, mode=1, tnear=tnear, tfar=tfar), rp >= 0)
            assert (rp >= 0).sum() > 100


def _deep(rng, levels=28, per=32, size=2.0, shrink=0.9):
    """Triangles whose hierarchy is a chain of `levels` nodes: each level halves
    the region and puts `per` slivers, boxes far larger than it that rays cross
    and seldom hit, into the half that the chain leaves, so that a node's
    children are those and the rest; at its end small wide triangles."""
    tris = []

    def put(c, s, wide=False):
        mid = rng.uniform(-1.0, 1.0, 3) if wide else rng.normal(size=3) * 1e-3
        p = np.array([[-1.0, -1.0, -1.0], [1.0, 1.0, 1.0], mid])
        tris.append(c + 0.5 * s * p * rng.choice([-1.0, 1.0], 3))

    ext = np.ones(3)
    for l in range(levels):
        ext[l % 3] *= 0.5
        base = np.zeros(3)
        base[l % 3] = ext[l % 3]
        for _ in range(per):
            put(base + rng.uniform(0.02, 0.98, 3) * ext, size * shrink ** l)
    for _ in range(per):
        put(rng.uniform(0.0, 1.0, 3) * ext, size * shrink ** levels, True)
    put(np.zeros(3), size * shrink ** levels)
    put(np.ones(3), size)
    v = np.concatenate(tris)
    return v, np.arange(len(v)).reshape(-1, 3)


def _deep_rays(rng, n):
    """Rays past the chain's end from everywhere."""
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    org = rng.uniform(-0.1, 0.1, (n, 3)) - d * rng.uniform(0.0, 3.0, (n, 1))
    return org.astype(np.float32), d.astype(np.float32)


@pytest.mark.parametrize("n", [64, 3001, 300001, 600000])
def test_deep_tree_queries(tmp_path, n):
    """A tree of 27 levels.  Where the rays outnumber the lanes, so that none
    are idle and take groups over, a lane's stack goes on past its LDS entries.
    The same rays from host arrays and from device arrays, whose scratch is the
    library's own and holds fewer lanes of so deep a tree."""
    rng = np.random.default_rng(n)
    v, f = _deep(rng)
    ctx, ref = _load(tmp_path, [dict(verts=v, faces=f)])
    with ctx:
        org, dirs = _deep_rays(rng, n)
        m = min(n, 20000)  # (brute force is for the first rays; all agree among themselves)
        t, u, w, p = ctx.trace_rays(org, dirs, 0)
        rt, ru, rw, rp = ref.closest(0, org[:m], dirs[:m], brute=True)
        assert np.array_equal(p[:m], rp) and np.array_equal(t[:m], rt)
        assert np.array_equal(u[:m], ru) and np.array_equal(w[:m], rw)
        assert np.array_equal(ctx.trace_rays(org, dirs, 0, mode=1), p >= 0)
        inf, eps = np.full(n, math.inf, np.float32), np.full(n, 0.001, np.float32)
        dt, du, dw, dp = _device_query(ctx, org, dirs, eps, inf, 0, 0)
        assert np.array_equal(dp, p) and np.array_equal(dt, t) and np.array_equal(du, u) and np.array_equal(dw, w)
        assert np.array_equal(_device_query(ctx, org, dirs, eps, inf, 1, 0)[3] != 0, p >= 0)


@pytest.fixture(scope="module")
def deep_scene(tmp_path_factory):
    d = str(tmp_path_factory.mktemp("deep"))
    rng = np.random.default_rng(2)
    doms = []
    for k in range(3):
        v, f = _deep(rng)
        doms.append(dict(verts=v + [k, 0.5, 0.0], faces=f, rgb=rng.integers(0, 256, (len(v), 3)).astype(np.uint8)))
    path = scenes.write_scene(d, "s", doms, ["light rect 0.5 4.4 0.5 2 0 0 0 0 2 4 4 4"])
    cam = dict(pos=[0.3, 0.7, 2.0], lookat=[0.0, 0.5, 0.0], up=[0.0, 1.0, 0.0], fov=8.0)
    kw = dict(image_w=640, image_h=480, pixel_samples=2, ao_mode=0, ao_samples=1, bounces=2, rr_start=3)
    ref = orc.Scene(path, d).render(nthreads=8, cam_pos=cam["pos"], cam_lookat=cam["lookat"], cam_up=cam["up"],
                                    fov=cam["fov"], **kw)
    return d, path, cam, kw, ref


@pytest.mark.parametrize("schedule,cache", [(0, -1), (1, -1), (0, 1), (1, 2)])
def test_deep_tree_frames(deep_scene, schedule, cache):
    """Such trees in a frame of more rays than lanes, resident and paged; the
    camera looks past the end of the first domain's chain."""
    import spray_amd as sa
    d, path, cam, kw, (rimg, rst) = deep_scene
    cfg = sa.default_config(has_camera=1, camera_pos=cam["pos"], camera_lookat=cam["lookat"], camera_up=cam["up"],
                            fov=cam["fov"], nthreads=8, schedule=schedule, **kw)
    with sa.Context(cfg) as ctx:
        if cache >= 0:
            ctx.set_cache_size(cache)
        ctx.load_scene(path, d)
        img, st = ctx.trace_frame()
    err = np.abs(img[..., :3] - rimg[..., :3])
    assert st["useful_rays"] == rst["useful_rays"] and st["final_hits"] == rst["final_hits"] > 10000
    assert math.sqrt(float((err ** 2).mean())) <= 1e-4 and float(err.max()) <= 1e-3
