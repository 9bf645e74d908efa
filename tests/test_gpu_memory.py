"""What a context keeps in HBM between calls, and what it gives back: the
frame's buffers while the schedule changes, scenes that leave little of the
HBM free or replace one another, meshes that grow from step to step, and the
images of paged domains."""
import ctypes as C
import os

import numpy as np
import pytest

import orc
import scenes
from test_gpu_edges import LIGHT, _cfg, _frame_ok, _sheet, _soup, lattices  # noqa: F401 (lattices: a fixture)

pytestmark = pytest.mark.gpu


def _hbm_blocks(least):
    """Device allocations of at least `least` bytes, as (address, bytes): the
    process's mappings of the GPU's device file."""
    out = set()
    for line in open("/proc/self/maps"):
        if "/dev/dri/" in line:
            a, b = (int(x, 16) for x in line.split()[0].split("-"))
            if b - a >= least:
                out.add((a, b - a))
    return out


def test_learned_frames_beside_batched_ones(lattices):  # noqa: F811
    """One context, batched and learned frames in turn: each as the oracle's,
    and a learned frame leaves the memory of the others where it is."""
    import spray_amd as sa
    d, ref = lattices
    kw = dict(image_w=160, image_h=120, pixel_samples=4, ao_mode=0, ao_samples=1, bounces=5, rr_start=3)
    with sa.Context(_cfg(schedule=1, **kw)) as ctx:
        ctx.load_scene(os.path.join(d, "g27.spray"), d)
        ctx.predictor_log(True, 200000)
        _frame_ok(ctx, ref["g27"], **kw)
        ctx.predictor_log(False)
        ctx.predictor_train(1, 1024, 2e-3)
        _frame_ok(ctx, ref["g27"], **kw)
        held = _hbm_blocks(32 << 20)
        for schedule in (2, 1, 2, 0, 2):
            ctx.set_schedule(schedule)
            _frame_ok(ctx, ref["g27"], **kw)
            if not held:
                pytest.skip("this driver does not show device allocations as mappings")
            assert held <= _hbm_blocks(32 << 20), schedule


class _Filler:
    """Device memory taken until only so much is free, from the HIP runtime the
    library itself links."""

    def __init__(self):
        self.rt = C.CDLL("libamdhip64.so.7")
        self.rt.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
        self.rt.hipFree.argtypes = [C.c_void_p]
        self.bufs = []

    def free_bytes(self):
        a, b = C.c_size_t(), C.c_size_t()
        assert self.rt.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
        return a.value

    def leave(self, want):
        for step in (64 << 30, 4 << 30, 256 << 20, 32 << 20):
            while self.free_bytes() - want > step:
                p = C.c_void_p()
                if self.rt.hipMalloc(C.byref(p), step) != 0:
                    break
                self.bufs.append(p)
        left = self.free_bytes() - want
        assert 0 <= left < 96 << 20, left

    def __enter__(self):
        return self

    def __exit__(self, *a):
        for p in self.bufs:
            self.rt.hipFree(p)
        self.bufs = []


def _retained(filler, scene):
    """HBM that a context holds once this scene is loaded."""
    import spray_amd as sa
    before = filler.free_bytes()
    with sa.Context(_cfg(image_w=16, image_h=12)) as ctx:
        ctx.scenegen_load("s", **scene)
        return before - filler.free_bytes()


def test_build_in_little_memory(lattices):  # noqa: F811
    """Four domains of 2 M triangles where the build's memory for one domain is
    free (0.34 GB), but not for four side by side."""
    import spray_amd as sa
    scene = dict(nx=4, ny=1, nz=1, res=300)
    with _Filler() as filler:
        need = _retained(filler, scene)
        with sa.Context(_cfg(image_w=16, image_h=12)) as ctx:
            filler.leave(need + (640 << 20))
            ctx.scenegen_load("s", **scene)
            rng = np.random.default_rng(1)
            d = rng.normal(size=(1000, 3)).astype(np.float32)
            org = (rng.uniform(0.2, 0.8, (1000, 3)) + [2.0, 0.0, 0.0]).astype(np.float32)
            _, _, _, few = ctx.trace_rays(org, d, 2)
    with sa.Context(_cfg(image_w=16, image_h=12)) as ctx:
        ctx.scenegen_load("s", **scene)
        assert np.array_equal(ctx.trace_rays(org, d, 2)[3], few) and (few >= 0).any()


def test_load_gets_idle_frame_memory(lattices):  # noqa: F811
    """The last scene's frame memory, kept for the next frames, makes room for
    what the next scene's build needs."""
    import spray_amd as sa
    d, _ = lattices
    scene = dict(nx=1, ny=1, nz=1, res=500)  # 5.5 M triangles, 0.9 GB of build memory
    with _Filler() as filler:
        need = _retained(filler, scene)
        with sa.Context(_cfg(schedule=1, image_w=1024, image_h=1024, pixel_samples=2, ao_samples=1, bounces=4)) as ctx:
            ctx.load_scene(os.path.join(d, "g2.spray"), d)
            before = filler.free_bytes()
            ctx.trace_frame(want_image=False)
            assert (2 << 30) < before - filler.free_bytes() < (4 << 30)  # (what a context keeps at most)
            ctx.load_scene(os.path.join(d, "g2.spray"), d)
            filler.leave(need + (320 << 20))
            ctx.scenegen_load("s", **scene)
            assert ctx.num_domains == 1


def test_smaller_scene_gives_memory_back(tmp_path, lattices):  # noqa: F811
    """After a scene of 0.4 GB, one of 0.15 GB holds what it needs alone."""
    import spray_amd as sa
    for name, res in (("large", 330), ("small", 200)):
        sa.scenegen_write(str(tmp_path), name, 1, 1, 1, res)
    with _Filler() as filler:
        held = []
        for names in (["small"], ["large", "small"]):
            before = filler.free_bytes()
            with sa.Context(_cfg(image_w=16, image_h=12)) as ctx:
                for name in names:
                    ctx.load_scene(os.path.join(str(tmp_path), name + ".spray"), str(tmp_path))
                held.append(before - filler.free_bytes())
        assert held[1] <= held[0] + (80 << 20), held


@pytest.mark.parametrize("schedule", [0, 1])
def test_growing_remeshes(schedule):
    """Remeshes whose pool outgrows its allocation again and again: every frame
    is that of a context that generated the step's mesh alone."""
    import spray_amd as sa
    kw = dict(image_w=48, image_h=36, pixel_samples=2, ao_mode=0, ao_samples=1, bounces=3, rr_start=3)
    scene = dict(nx=2, ny=2, nz=1, res=20, rgb=0xB3B3B3, extra_lines=LIGHT)
    most, grown = 0, 0
    with sa.Context(_cfg(schedule=schedule, **kw)) as ctx:
        ctx.scenegen_load("s", **scene)
        for phase in (0.0, 0.25, 0.5, 0.75, 1.0, 0.25, 2.25):
            ctx.remesh(phase)
            tris = sum(ctx.mesh_size(d)[1] for d in range(4))
            grown += tris > most
            most = max(most, tris)
            img, st = ctx.trace_frame()
            with sa.Context(_cfg(schedule=schedule, **kw)) as alone:
                alone.scenegen_load("s", phase=phase, **scene)
                want, wst = alone.trace_frame()
                assert all(np.array_equal(ctx.normals(d), alone.normals(d)) for d in range(4)), phase
            assert all(st[k] == wst[k] for k in ("useful_rays", "final_hits", "shades")), phase
            assert np.abs(img - want).max() <= 1e-5, phase
    assert grown >= 5


@pytest.mark.parametrize("schedule", [0, 1])
@pytest.mark.parametrize("cache", [2, 5])
def test_paged_shading_of_both_forms(tmp_path, cache, schedule):
    """Domains with shared vertices, whose mesh crosses the host link, and
    without, whose shading records do, every vertex of a colour of its own."""
    import spray_amd as sa
    rng = np.random.default_rng(4)
    doms = []
    for d in range(6):
        v, f = _sheet(rng, 13) if d % 2 else _soup(rng, 1 if d == 4 else 211, 0.2)
        doms.append(dict(verts=v + [d % 3, d // 3, 1.0], faces=f,
                         rgb=rng.integers(0, 256, (len(v), 3)).astype(np.uint8)))
    path = scenes.write_scene(str(tmp_path), "s", doms, [LIGHT])
    kw = dict(image_w=90, image_h=70, pixel_samples=2, ao_mode=0, ao_samples=1, bounces=3, rr_start=3)
    with sa.Context(_cfg(schedule=schedule, **kw)) as ctx:
        ctx.set_cache_size(cache)
        ctx.load_scene(path, str(tmp_path))
        ref = orc.Scene(path, str(tmp_path))
        for _ in range(2):
            _frame_ok(ctx, ref, **kw)
        assert ctx.cache_state()[3] > 6  # (misses)
