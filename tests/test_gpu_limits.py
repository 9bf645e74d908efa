"""The trace kernels at the limits of a ray and of a tree, against the oracle's
brute force over every triangle (bit for bit, as the hits use its arithmetic):
hits behind a ray's origin."""
import math

import numpy as np
import pytest

from test_gpu_edges import _load, _rays_at, _soup

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
