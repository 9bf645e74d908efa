"""What a context keeps in HBM between calls, and what it gives back: the
frame's buffers while the schedule changes."""
import os

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
