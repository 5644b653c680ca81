"""Draws that share their geometry, split into setup groups by how much work
the frame holds: from pairs on small frames to sixteen draws a group on large
ones, larger groups first, lists of 1 to 48 views, every view against the
oracle's render of the frame."""
import math

import numpy as np
import pytest

from softrast_amd import scenes
from tests import helpers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nviews,spheres,ndraws", [(1, 8, 2), (2, 8, 2), (3, 8, 1), (5, 40, 3), (17, 60, 2), (13, 700, 1),
                                                   (48, 1000, 1), (48, 1500, 2)])
def test_setup_groups(nviews, spheres, ndraws):
    import softrast_amd as sr
    w, h = 96, 64
    s = scenes.spheres_scene(70 + nviews, spheres, ndraws, w, h, tex_size=0)
    tex = [sr.TextureData().CreateFromRGBA8(scenes.value_noise_rgba8(5, 64, 64), 64, 64, True)]
    for d in s.draws:
        d.texture = 0
    own = scenes.spheres_scene(700 + nviews, 3, 1, w, h, tex_size=0).draws[0]  # a draw that no other view has
    own.texture = 0
    views = []
    for k in range(nviews):
        t = math.radians((k - (nviews - 1) / 2.0) * 0.5)
        mvp = scenes.camera_mvp((0.0, 0.0, 0.0), (math.sin(t), 0.0, math.cos(t)), 60.0, w / h)
        views.append(scenes.Scene(w, h, mvp, list(s.draws) + ([own] if k == nviews // 2 else []), [], {}))
    vs = scenes.ViewSet(views, [])
    print(f"[groups] views={nviews} tris={vs.num_tris}", flush=True)
    planes, _ = helpers.oracle_render_views(vs, tex)
    ctx = sr.RenderContext(flags=sr.CFG_KEEP_PRIMID)
    fbs = [sr.FrameBuffer(ctx, w, h) for _ in views]
    helpers.gpu_render_views(vs, tex, ctx, fbs)
    for k, (fb, p) in enumerate(zip(fbs, planes)):
        col, dep, pid = fb.read_tiles(primid=True)
        assert not any(helpers.compare(p, col.reshape(-1), dep.reshape(-1), pid.reshape(-1)).values()), k
    for fb in fbs:
        fb.destroy()
    ctx.Shutdown()
