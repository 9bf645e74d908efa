"""What a context keeps in HBM between calls, and what it gives back: the
frame's buffers while the schedule changes, and scenes that leave little of
the HBM free or replace one another."""
import ctypes as C
import os

import numpy as np
import pytest

from test_gpu_edges import _cfg, _frame_ok, lattices  # noqa: F401 (lattices: a fixture)

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
