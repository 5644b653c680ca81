"""Binning of primitives that span many work bins: the walk that takes one
primitive at a time (64 candidate bins and more) beside the compacted walk of
small ones, from the set-up and from the clipper, against the oracle."""
import numpy as np
import pytest

from softrast_amd import scenes
from tests import helpers

pytestmark = pytest.mark.gpu

# spans in 8-pixel bins: 1, 4, 60, 63, 64, 65, 128, 252, 256, 260 candidates, a whole row, the whole picture
SPANS = ((1, 1), (2, 2), (10, 6), (9, 7), (8, 8), (13, 5), (16, 8), (28, 9), (16, 16), (26, 10), (63, 2), (63, 63))


def _scene(seed, size, clipped):
    rng = np.random.default_rng(seed)
    tris = []
    for w, h in SPANS:
        for k in range(6):
            bx, by = rng.integers(0, size // 8 - w + 1), rng.integers(0, size // 8 - h + 1)
            x0, y0 = bx * 8 + rng.uniform(0.5, 7), by * 8 + rng.uniform(0.5, 7)
            x1, y1 = (bx + w) * 8 - rng.uniform(0.5, 1.5), (by + h) * 8 - rng.uniform(0.5, 1.5)
            third = ((x0, y1), (x1, y1), (x0 + 1.0, y0 + 1.0))[k % 3]  # half the box, the other half, a sliver along it
            t = [(x0, y0), (x1, y0 if k % 3 < 2 else y1), third]
            if clipped and k % 2:
                t[k // 2] = (t[k // 2][0] + rng.choice([-1, 1]) * 1.3 * size, t[k // 2][1])
            tris += [t, t[::-1]]
    p = np.array(tris, np.float64).reshape(-1, 2) * 2.0 / size - 1.0
    v = np.zeros((len(p), 8), np.float32)
    v[:, 0], v[:, 1] = p[:, 0], -p[:, 1]
    v[:, 2] = rng.uniform(0.1, 0.9, len(p))
    v[:, 6:8] = rng.uniform(-2, 2, (len(p), 2))
    order = rng.permutation(len(p) // 3)  # big and small ones mixed in a wave
    idx = np.arange(len(p), dtype=np.uint32).reshape(-1, 3)[order].reshape(-1).copy()
    tex = [rng.integers(0, 256, (64, 64, 4), dtype=np.uint8)]
    return scenes.Scene(size, size, np.eye(4, dtype=np.float32).reshape(-1),
                        [scenes.Draw(v.view(scenes.VERTEX_DTYPE).reshape(-1), idx, 0)], tex, {})


@pytest.mark.parametrize("clipped", [False, True])
@pytest.mark.parametrize("bin_size", [8, 16, 32])
def test_many_bin_primitives(bin_size, clipped):
    sc = _scene(40 + bin_size, 504, clipped)
    print(f"[bins] bin_size={bin_size} clipped={clipped} tris={sc.num_tris}", flush=True)
    tex = helpers.build_textures(sc)
    ref, rstats = helpers.oracle_render(sc, tex, nthreads=4)
    col, dep, pid, gstats = helpers.gpu_render(sc, tex, bin_size=bin_size)
    assert not any(helpers.compare(ref, col, dep, pid).values())
    assert gstats["frags_raster"] == rstats["frags_raster"] and gstats["bin_entries"] == rstats["bin_entries"]
    assert (gstats["tris_clipped"] > 0) == clipped
