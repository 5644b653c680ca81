"""The clipper's queue, kept as lists of 256-triangle chunks: frames whose
draws end inside a chunk, at its edge and past a whole round of lists, most
triangles crossing a side of the frustum, against the oracle."""
import numpy as np
import pytest

from softrast_amd import scenes
from tests import helpers

pytestmark = pytest.mark.gpu


def _scene(seed, counts, size):
    rng = np.random.default_rng(seed)
    draws = []
    for n in counts:
        centre = rng.choice([-1.0, 1.0], (n, 1, 2)) * rng.uniform(0.9, 1.1, (n, 1, 2))  # on the picture's corners
        p = centre * rng.permuted(np.tile([1.0, 0.3], (n, 1, 1)), axis=2) + rng.normal(0, 0.08, (n, 3, 2))
        v = np.zeros((3 * n, 8), np.float32)
        v[:, :2] = p.reshape(-1, 2)
        v[:, 2] = rng.uniform(0.1, 0.9, 3 * n)
        v[:, 6:8] = rng.uniform(-2, 2, (3 * n, 2))
        draws.append(scenes.Draw(v.view(scenes.VERTEX_DTYPE).reshape(-1), np.arange(3 * n, dtype=np.uint32), 0))
    tex = [rng.integers(0, 256, (64, 64, 4), dtype=np.uint8)]
    return scenes.Scene(size, size, np.eye(4, dtype=np.float32).reshape(-1), draws, tex, {})


@pytest.mark.parametrize("counts", [(1,), (255,), (256,), (257,), (63, 130, 5, 300), (4095, 2), (4096, 1), (4097, 31, 700),
                                    (97,) * 60, (20000,)])
def test_clip_lists(counts):
    sc = _scene(900 + len(counts) + counts[0], counts, 192)
    print(f"[clip] counts={counts[:4]}", flush=True)
    tex = helpers.build_textures(sc)
    ref, rstats = helpers.oracle_render(sc, tex, nthreads=4)
    col, dep, pid, gstats = helpers.gpu_render(sc, tex)
    assert not any(helpers.compare(ref, col, dep, pid).values())
    assert gstats["frags_raster"] == rstats["frags_raster"] and gstats["bin_entries"] == rstats["bin_entries"]
    assert sum(counts) < 8 or gstats["tris_clipped"] > sum(counts) // 8
