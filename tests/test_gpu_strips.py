"""How a small frame's 32-pixel bins are split into strips where the
configuration leaves it open, and the split frames against the oracle: frames
below, at and above the limits of a two-plane frame, a SponzaShader frame, a
statistics frame and configured workgroups per CU."""
import pytest

from softrast_amd import scenes
from tests import helpers

pytestmark = pytest.mark.gpu

# (width, height): 60, 64, 240, 256, 540, 704, 768, 816 bins
CASES = [
    (320, 180, 0, False, 0, 4), (960, 540, 0, False, 0, 2), (1024, 768, 0, False, 0, 2), (1088, 768, 0, False, 0, 1),
    (320, 180, 3, False, 0, 4), (960, 540, 3, False, 0, 2), (1024, 704, 3, False, 0, 2), (1088, 768, 3, False, 0, 1),
    (256, 256, 0, True, 0, 4), (640, 360, 0, True, 0, 1), (512, 512, 3, True, 0, 1), (960, 540, 0, True, 0, 1),
    (320, 180, 0, False, 1, 4), (640, 360, 0, False, 1, 1), (640, 360, 0, False, 2, 2), (960, 540, 0, False, 2, 1),
]


@pytest.mark.parametrize("width,height,shader,stats,wg_per_cu,strips", CASES)
def test_strips_by_frame(width, height, shader, stats, wg_per_cu, strips):
    import softrast_amd as sr
    print(f"[strips] {width}x{height} shader={shader} stats={stats} wg_per_cu={wg_per_cu}", flush=True)
    sc = helpers.random_scene(600 + width + height, 1500, width, height, clip_heavy=True, shaders=(shader,))
    tex = helpers.build_textures(sc)
    kw = dict(sponza=sr.SponzaConstants(sun_dir=(0.0, 1.0, 0.0), ambient=(0.3, 0.3, 0.3))) if shader == 3 else {}
    ref, rstats = helpers.oracle_render(sc, tex, nthreads=8, **kw)
    flags = sr.CFG_KEEP_PRIMID | (sr.CFG_STATS if stats else 0)
    col, dep, pid, st = helpers.gpu_render(sc, tex, flags=flags, wg_per_cu=wg_per_cu, **kw)
    assert not any(helpers.compare(ref, col, dep, pid).values())
    assert st["bin_size"] == 32 and st["wg_per_tile"] == strips
    assert not stats or st["frags_raster"] == rstats["frags_raster"]
