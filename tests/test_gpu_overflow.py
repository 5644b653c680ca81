"""Frames without statistics and learned order, whose counters the scan hands
to the host (one launch for up to 4,096 bins, three above): an arena that
overflows is seen and the frame rendered again, an index out of range is an
error, and the frame after it is right, launched one by one, as a graph and by
the non-allocating EndFrame."""
import pytest

from tests import helpers

pytestmark = pytest.mark.gpu

SRG_ERR_INDEX_RANGE = -4


@pytest.mark.parametrize("how", ["launched", "graph", "noalloc"])
@pytest.mark.parametrize("bin_size", [32, 8])
def test_counters_from_the_scan(bin_size, how):
    import softrast_amd as sr
    flags = sr.CFG_KEEP_PRIMID | (sr.CFG_GRAPH if how == "graph" else 0)
    noalloc = how == "noalloc"
    sc = helpers.random_scene(810 + bin_size, 6000, 640, 512, clip_heavy=True)  # 320 bins of 32 pixels, 5,120 of 8
    tex = helpers.build_textures(sc)
    ref, rstats = helpers.oracle_render(sc, tex, nthreads=8)
    ctx = sr.RenderContext(flags=flags, bin_size=bin_size, max_prims=1, max_entries=1)
    fb = sr.FrameBuffer(ctx, sc.width, sc.height)

    def check(st):
        col, dep, pid = fb.read_tiles(primid=True)
        assert not any(helpers.compare(ref, col.reshape(-1), dep.reshape(-1), pid.reshape(-1)).values())
        assert st["tris_clipped"] > 0 and st["tris_in"] == sc.num_tris and st["work_entries"] > 0

    for frame in range(3):
        print(f"[overflow] {how} bin_size={bin_size} frame={frame}", flush=True)
        st = helpers.gpu_render(sc, tex, ctx=ctx, fb=fb, noalloc=noalloc)
        check(st)
        # the grown arenas are kept; the non-allocating EndFrame's records are carved anew each time
        assert (st["retries"] > 0) == (frame == 0 or noalloc), (frame, st["retries"])

    good = sc.draws[0].indices
    sc.draws[0].indices = good.copy()
    sc.draws[0].indices[777] = len(sc.draws[0].vertices)
    print(f"[overflow] {how} bin_size={bin_size} index out of range", flush=True)
    with pytest.raises(sr.SrgError) as e:
        helpers.gpu_render(sc, tex, ctx=ctx, fb=fb, noalloc=noalloc)
    assert e.value.status == SRG_ERR_INDEX_RANGE
    sc.draws[0].indices = good
    check(helpers.gpu_render(sc, tex, ctx=ctx, fb=fb, noalloc=noalloc))
    fb.destroy()
    ctx.Shutdown()
