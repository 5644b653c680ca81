"""Asynchronous blits on both sides of the size up to which the de-tile kernel
writes page-locked memory itself, back to back on both planes, from pageable and
page-locked memory of every caching kind: the bytes, and nothing beside them,
are there when the callback runs."""
import ctypes

import numpy as np
import pytest

from tests.test_gpu_blit import GUARD, _hip

pytestmark = pytest.mark.gpu

# hipHostMalloc: default, write-combined, coherent, non-coherent
FLAGS = (0x0, 0x4, 0x40000000, 0x80000000)


@pytest.mark.parametrize("width,height", [(1, 1), (63, 65), (128, 64), (8192, 1), (129, 64), (8193, 1), (321, 180)])
def test_async_blit_sizes(width, height):
    import softrast_amd as sr
    ctx = sr.RenderContext()
    hip = _hip()
    fb = sr.FrameBuffer(ctx, width, height)
    n = width * height * 4
    locked = []
    buffers = [("pageable", np.empty(n + 2 * GUARD, np.uint8))]
    for f in FLAGS:
        p = ctypes.c_void_p()
        assert hip.hipHostMalloc(ctypes.byref(p), n + 2 * GUARD, f) == 0
        locked.append(p)
        buffers.append((f"{f:#x}", np.ctypeslib.as_array((ctypes.c_uint8 * (n + 2 * GUARD)).from_address(p.value))))
    rng = np.random.default_rng(width * 8209 + height)
    for name, whole in buffers:
        print(f"[blit_async] {width}x{height} {name}", flush=True)
        for step in range(6):
            tiles = rng.integers(0, 1 << 32, (fb.tiles_y * fb.tiles_x, 64, 64), dtype=np.uint64).astype(np.uint32)
            rows = tiles.reshape(fb.tiles_y, fb.tiles_x, 64, 64).transpose(0, 2, 1, 3)
            rows = np.ascontiguousarray(rows.reshape(fb.tiles_y * 64, fb.tiles_x * 64)[:height, :width])
            fb.write_tiles(tiles, np.zeros(tiles.shape, np.float32))
            whole[:] = 0x5A
            out = whole[GUARD:GUARD + n]
            seen = []
            ctx.BlitAsync(fb, out, onFinish=lambda _u: seen.append(out.copy()), bgra=step % 2 == 1)
            # the planes are swapped: the next write goes to the other one while the blit runs
            fb.write_tiles(np.full_like(tiles, step), np.zeros(tiles.shape, np.float32))
            ctx.BlitWait(fb)
            want = rows if step % 2 == 0 else (rows & 0xFF00FF00) | ((rows >> 16) & 0xFF) | ((rows & 0xFF) << 16)
            want = want.view(np.uint8).reshape(-1)
            assert len(seen) == 1 and np.array_equal(seen[0], want) and np.array_equal(out, want)
            assert (whole[:GUARD] == 0x5A).all() and (whole[GUARD + n:] == 0x5A).all()
    fb.destroy()
    for p in locked:
        hip.hipHostFree(p)
    ctx.Shutdown()
