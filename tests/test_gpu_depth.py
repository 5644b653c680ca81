"""Depth planes that are not finite, beside ordinary ones in the same waves:
triangles whose vertices are collinear in floating point, so that the plane
divides by 0, but not after snapping to 1/256 pixel, so that they are not
culled; and depth buffers that hold NaN, infinities, zeros and negatives."""
import numpy as np
import pytest

from softrast_amd import scenes
from tests import helpers

pytestmark = pytest.mark.gpu
SIZE = 256  # viewport: pixel = 128 +- 128 * clip, exact for multiples of 2^-23


def _scene(seed):
    rng = np.random.default_rng(seed)
    tris, zs = [], []
    for k in range(3000):
        if k % 3:  # p0 + t * d through pixel centres, t in steps of 2^-12: exact, collinear
            p0 = rng.integers(20, 200, 2)
            d = rng.integers(-8, 9, 2)
            t = np.sort(rng.integers(0, 4 * 4096, 3)) / 4096.0
            tri = [p0 + x * d for x in t]
            if k % 2:
                tri = tri[::-1]
        else:
            tri = list(rng.uniform(5, 250, 2) + rng.normal(0, 9, (3, 2)))
        tris.append(tri)
        zs.append(rng.uniform(0.05, 0.95, 3) if k % 5 else np.full(3, 0.5))
    p = np.array(tris).reshape(-1, 2)
    v = np.zeros((len(p), 8), np.float32)
    v[:, 0], v[:, 1] = (p[:, 0] - 128) / 128, (128 - p[:, 1]) / 128
    v[:, 2] = np.array(zs).reshape(-1)
    v[:, 6:8] = rng.uniform(-2, 2, (len(p), 2))
    v[::17, 6], v[::29, 7], v[::13, 6] = np.inf, np.nan, 3e38  # texture coordinates that are not finite either
    tex = [rng.integers(0, 256, (64, 64, 4), dtype=np.uint8)]
    return scenes.Scene(SIZE, SIZE, np.eye(4, dtype=np.float32).reshape(-1),
                        [scenes.Draw(v.view(scenes.VERTEX_DTYPE).reshape(-1), np.arange(len(p), dtype=np.uint32), 0)], tex, {})


@pytest.mark.parametrize("init", [False, True])
@pytest.mark.parametrize("bin_size", [8, 32, 64])
def test_depth_not_finite(bin_size, init):
    sc = _scene(7 + bin_size)
    plane = None
    if init:
        rng = np.random.default_rng(3)
        depth = rng.choice(np.array([0.0, -0.0, -1.0, 0.3, 1e-40, np.inf, -np.inf, np.nan], np.float32), (16, 64, 64))
        plane = (np.zeros((16, 64, 64), np.uint32), depth)
    print(f"[depth] bin_size={bin_size} init={init}", flush=True)
    tex = helpers.build_textures(sc)
    kw = dict(clear=None, plane_init=plane) if init else {}
    ref, rstats = helpers.oracle_render(sc, tex, nthreads=4, **kw)
    assert rstats["frags_raster"] - rstats["frags_passed"] > 500  # collinear ones cover pixels and never win
    col, dep, pid, gstats = helpers.gpu_render(sc, tex, bin_size=bin_size, **kw)
    d = helpers.compare(ref, col, dep, pid)
    print(f"[depth] diffs {d} covered {int((pid != 0xFFFFFFFF).sum())} not finite {int((~np.isfinite(dep)).sum())}", flush=True)
    assert not any(d.values())
    assert gstats["frags_raster"] == rstats["frags_raster"]
