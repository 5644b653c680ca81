"""Textures whose rows are made in two batches, level 1 after the others in the
same workspace, beside the largest that are made in one: the bytes equal the
host build's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(2048, 2048), (4096, 2048), (1024, 8192), (8192, 1024)])
def test_device_mips_in_batches(w, h):
    import softrast_amd as sr
    print(f"[texture] case=batches size={w}x{h}", flush=True)
    img = np.random.default_rng(w * 3 + h).integers(0, 256, (h, w, 4), dtype=np.uint8)
    img[:, 0], img[:, -1], img[0], img[-1] = 255, 0, 255, 0
    host = sr.TextureData().CreateFromRGBA8(img, w, h, True)
    ctx = sr.RenderContext()
    for _ in range(2):
        dev = ctx.CreateTexture(img, w, h, True).read()
        assert np.array_equal(dev.m_texels, host.m_texels) and dev.m_numMips == host.m_numMips
    ctx.Shutdown()
