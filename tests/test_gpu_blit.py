"""Pixels to the caller's memory: Blit, BlitAsync and read_tiles write the same
bytes, and nothing beside them, whether the memory is pageable (through
page-locked chunks), page-locked (written by the kernel) or not word-aligned."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# one row, one tile, partial tiles, one chunk, rows that do not divide a chunk, several chunks
SIZES = ((1, 1), (64, 64), (65, 63), (257, 130), (1000, 263), (1021, 770), (1920, 1080))
GUARD = 64


def _hip():
    """The HIP runtime that the library itself uses."""
    with open("/proc/self/maps") as f:
        path = next(line.split()[-1] for line in f if "libamdhip64" in line)
    hip = ctypes.CDLL(path)
    hip.hipHostMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t, ctypes.c_uint]
    hip.hipHostFree.argtypes = [ctypes.c_void_p]
    return hip


@pytest.mark.parametrize("width,height", SIZES)
def test_blit_targets(width, height):
    import softrast_amd as sr
    ctx = sr.RenderContext()
    hip = _hip()
    fb = sr.FrameBuffer(ctx, width, height)
    rng = np.random.default_rng(width * 4099 + height)
    tiles = rng.integers(0, 1 << 32, (fb.tiles_y * fb.tiles_x, 64, 64), dtype=np.uint64).astype(np.uint32)
    depth = rng.uniform(0.0, 1.0, tiles.shape).astype(np.float32)
    rows = tiles.reshape(fb.tiles_y, fb.tiles_x, 64, 64).transpose(0, 2, 1, 3).reshape(fb.tiles_y * 64, fb.tiles_x * 64)
    rows = np.ascontiguousarray(rows[:height, :width])
    swapped = (rows & 0xFF00FF00) | ((rows >> 16) & 0xFF) | ((rows & 0xFF) << 16)
    size = 2 * GUARD + 1 + rows.nbytes
    locked = ctypes.c_void_p()
    assert hip.hipHostMalloc(ctypes.byref(locked), size, 0) == 0
    buffers = {"pageable": np.empty(size, np.uint8),
               "pinned": np.ctypeslib.as_array((ctypes.c_uint8 * size).from_address(locked.value))}
    for kind in ("pageable", "pinned", "pageable_unaligned", "pinned_unaligned"):
        for call in ("blit", "async", "async_bgra"):
            print(f"[blit] {width}x{height} {kind} {call}", flush=True)
            fb.write_tiles(tiles, depth)
            got_c, got_d = fb.read_tiles()
            assert np.array_equal(got_c, tiles) and np.array_equal(got_d, depth)
            whole, lead = buffers[kind.split("_")[0]], GUARD + (1 if kind.endswith("unaligned") else 0)
            whole[:] = 0xA5
            out = whole[lead:lead + rows.nbytes]
            if call == "blit":
                ctx.Blit(fb, out)
            else:
                ctx.BlitAsync(fb, out, bgra=call == "async_bgra")
                ctx.BlitWait(fb)
            assert np.array_equal(out, (swapped if call == "async_bgra" else rows).view(np.uint8).reshape(-1))
            assert (whole[:lead] == 0xA5).all() and (whole[lead + rows.nbytes:] == 0xA5).all()
    fb.destroy()
    hip.hipHostFree(locked)
    ctx.Shutdown()
