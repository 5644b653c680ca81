"""What a program does with this renderer, as cases that can be timed.

A pass is one frame (or one batch of views) through the Python mirror of the C
ABI, from BeginFrame to the pixels in the program's own host memory: clear,
draw list, EndFrame, then Blit of every framebuffer (the only way an image
leaves the library), or one of the other two read paths. Framebuffers, vertex
buffers, textures and the prepared draw list are what a program keeps between
frames. One case builds a texture instead, the other work that a program hands
to the GPU. Every output is whole numbers: RGBA8 words, the bits of the depth
plane, texture bytes; the renderer's contract is that they are exact.
"""
import math
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

import softrast_amd as sr
from softrast_amd import scenes


def listed():
    return [
        # the smallest frame: 3,072 triangles at 320x180, a thumbnail or a preview window; pageable target
        dict(name="cubes_320x180", kind="cubes", grid=16, width=320, height=180, tex=128, pinned=False),
        # the viewer's first scene: 12,288 triangles with u16 indices at 1280x720
        dict(name="cubes_720p", kind="cubes", grid=32, width=1280, height=720, tex=512, pinned=True),
        # the ordinary heavy frame: 1 M triangles at 1080p in 8 textured draws
        dict(name="spheres_1080p_1m", kind="spheres", spheres=4000, draws=8, views=1, width=1920, height=1080, tex=2048,
             shader="unlit", order=0, graph=False, pinned=True),
        # the viewer's lit scene shader: 16 point lights per pixel, 250 k triangles
        dict(name="sponza_1080p_250k", kind="spheres", spheres=1000, draws=4, views=1, width=1920, height=1080,
             tex=1024, shader="sponza", order=0, graph=False, pinned=True),
        # image sets for training: 64 small views of one scene in one EndFrame
        dict(name="views64_512_100k", kind="spheres", spheres=400, draws=2, views=64, width=512, height=512, tex=1024,
             shader="unlit", order=1, graph=True, pinned=True),
        # the batched path in full: several 1080p cameras on 1 M triangles, learned queue order
        dict(name="views12_1080p_1m", kind="spheres", spheres=4000, draws=8, views=12, width=1920, height=1080, tex=2048,
             shader="unlit", order=2, graph=True, pinned=True),
        # independent requests gathered into one frame: sizes 256^2 to 1080p, 1 k to 500 k triangles each
        dict(name="mixed_24_views", kind="mixed", views=24, tex=1024, pinned=True),
        # a crowded 4K frame: 90% of 2 M triangles in a tenth of the picture, 0.5 to 2000 px^2 each
        dict(name="clustered_4k_2m", kind="clustered", views=1, tris=2000000, width=3840, height=2160, tex=2048,
             clustered=0.9, parts=2, pinned=True),
        # a batch of views without common geometry, 1440p, 1 M triangles each
        dict(name="combined_4x1440p_1m", kind="clustered", views=4, tris=1000000, width=2560, height=1440, tex=2048,
             clustered=0.5, parts=1, pinned=True),
        # a camera inside the geometry: most triangles cross the frustum; the non-allocating EndFrame of a serving
        # loop, normals shown, colour and depth tiles read
        dict(name="inside_960x540_60k", kind="inside", tris=60000, width=960, height=540, shader="normals"),
        # an interactive window: each frame is presented as BGRA while the next one renders
        dict(name="present_1080p_250k", kind="present", spheres=1000, draws=4, width=1920, height=1080, tex=1024),
        # loading: one 1024^2 RGBA8 image to a tiled texture with all its mips, kept as the loader's cache keeps it
        dict(name="texture_1024", kind="texture", width=1024, height=1024),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["cubes", "spheres", "views", "mixed", "clustered", "inside", "present", "texture"])
    width, height = rng.randint(160, 1920), rng.randint(90, 1080)
    tex = 1 << rng.randint(7, 11)
    if kind == "cubes":
        return dict(kind="cubes", grid=rng.randint(4, 37), width=width, height=height, tex=tex, pinned=rng.random() < 0.5)
    if kind == "spheres":
        return dict(kind="spheres", spheres=_log(rng, 20, 4000), draws=rng.randint(1, 8), views=1, width=width, height=height,
                    tex=tex, shader=rng.choice(["unlit", "unlit", "sponza", "normals", "uvs"]), order=rng.randint(0, 2),
                    graph=rng.random() < 0.5, pinned=rng.random() < 0.7)
    if kind == "views":
        side = rng.randint(96, 768)
        return dict(kind="spheres", spheres=_log(rng, 40, 800), draws=rng.randint(1, 4), views=rng.randint(2, 48), width=side,
                    height=rng.randint(96, 768), tex=tex, shader="unlit", order=rng.randint(0, 2), graph=True, pinned=True)
    if kind == "mixed":
        return dict(kind="mixed", views=rng.randint(3, 24), tex=tex, pinned=True)
    if kind == "clustered":
        return dict(kind="clustered", views=rng.randint(1, 2), tris=_log(rng, 20000, 800000), width=rng.randint(640, 2560),
                    height=rng.randint(360, 1440), tex=tex, clustered=rng.choice([0.0, 0.5, 0.9]), parts=rng.choice([1, 2]),
                    pinned=True)
    if kind == "inside":
        return dict(kind="inside", tris=_log(rng, 500, 60000), width=rng.randint(160, 960), height=rng.randint(90, 540),
                    shader=rng.choice(["normals", "uvs", "unlit"]))
    if kind == "present":
        return dict(kind="present", spheres=_log(rng, 20, 1000), draws=rng.randint(1, 4), width=width, height=height, tex=tex)
    return dict(kind="texture", width=1 << rng.randint(5, 11), height=1 << rng.randint(5, 10))


# ---- inputs ----

def _noise(seed, width, height):
    """Value noise, RGBA8 (height, width, 4): four octaves of smoothed random grids, as photographs and painted
    textures have detail at every scale."""
    g = torch.Generator().manual_seed(seed)
    out = torch.zeros(1, 4, height, width, device="cuda")
    for k, cells in enumerate((8, 32, 128, 512)):
        grid = torch.rand(1, 4, min(cells, height), min(cells, width), generator=g).cuda()
        out += torch.nn.functional.interpolate(grid, size=(height, width), mode="bilinear", align_corners=False) / (1 << k)
    out = (out * (255.0 / 1.875)).round().clamp(0, 255).to(torch.uint8)
    return np.ascontiguousarray(out[0].permute(1, 2, 0).cpu().numpy())


def _host(shape, pinned):
    """Where the pixels go: memory that the program allocated once, page-locked where it cares about the copy."""
    return torch.empty(shape, dtype=torch.int32, pin_memory=pinned).numpy()


_SHADERS = {"unlit": sr.UnlitDiffuseShader, "normals": sr.VisualizeNormalsShader, "uvs": sr.VisualizeUVsShader,
            "sponza": sr.SponzaShader}


def _call(fb, d, mvp, shader, tex):
    c = sr.DrawCall().SetFrameBuffer(fb).SetMVP(mvp).SetPixelShader(_SHADERS[shader], tex)
    c.SetIndexBuffer(d.indices, d.indices.dtype.itemsize, len(d.indices))
    c.SetPositionBuffer(d.vertices, 32, len(d.vertices))
    return c.SetAttributeBuffer(d.vertices, 32, len(d.vertices), 6)


def _inside_scene(seed, ntris, width, height):
    """Triangles all around a camera at the origin, sizes log-normal, both windings: many reach behind the near plane
    or out of the sides."""
    rng = np.random.default_rng(seed)
    centre = np.stack([rng.uniform(-26, 26, ntris), rng.uniform(-15, 15, ntris), rng.uniform(-4, 30, ntris)], 1)
    size = np.exp(rng.normal(-0.5, 1.0, ntris))[:, None, None]
    v = np.zeros((ntris * 3, 8), np.float32)
    v[:, :3] = (centre[:, None, :] + rng.normal(0, 1, (ntris, 3, 3)) * size).reshape(-1, 3)
    n = rng.normal(0, 1, (ntris * 3, 3))
    v[:, 3:6] = n / np.linalg.norm(n, axis=1, keepdims=True)
    v[:, 6:] = rng.uniform(-3, 3, (ntris * 3, 2))
    mvp = scenes.camera_mvp((0.0, 0.0, 0.0), (0.0, 0.0, 1.0), 60.0, width / height)
    idx = np.arange(ntris * 3, dtype=np.uint32)
    return scenes.Draw(v.view(scenes.VERTEX_DTYPE).reshape(-1), idx, 0), mvp


def _views(case, seed):
    """The views of a pass: a list of (width, height, mvp, draws)."""
    kind = case["kind"]
    if kind == "cubes":
        v, i = scenes.cube_grid_mesh(seed, case["grid"], case["grid"])
        if len(v) <= 0x10000:
            i = i.astype(np.uint16)
        mvp = scenes.camera_mvp((0.0, 8.0, -20.0), (0.0, 0.0, 0.0), 60.0, case["width"] / case["height"])
        return [(case["width"], case["height"], mvp, [scenes.Draw(v, i, 0)])]
    if kind in ("spheres", "present"):
        s = scenes.spheres_scene(seed, case["spheres"], case["draws"], case["width"], case["height"], tex_size=0)
        for k, d in enumerate(s.draws):
            d.texture = k
        views = case.get("views", 1)
        out = []
        for k in range(views):  # cameras turned by up to 2 degrees each way
            t = math.radians((k - (views - 1) / 2.0) * 4.0 / max(1, views - 1))
            mvp = scenes.camera_mvp((0.0, 0.0, 0.0), (math.sin(t), 0.0, math.cos(t)), 60.0, case["width"] / case["height"])
            out.append((case["width"], case["height"], mvp, s.draws))
        return out
    if kind == "mixed":  # the sizes in turn, triangle counts evenly over the logarithm, spheres from none to all
        n, out = case["views"], []
        for k in range(n):
            w, h = scenes.MIXED_RESOLUTIONS[k % len(scenes.MIXED_RESOLUTIONS)]
            tris = int(round(1000 * 500 ** (((5 * k + 2) % n + 0.5) / n)))
            v = scenes.shape_mix_view(seed + 31 * k, tris, w, h, ((3 * k + 1) % n) / n, (k % 4, (k + 1) % 4))
            out.append((w, h, v.mvp, v.draws))
        return out
    if kind == "clustered":
        def one(k):
            s = scenes.clustered_scene(seed + 7919 * k, case["tris"], case["width"], case["height"], ndraws=4, tex_size=0,
                                       clustered=case["clustered"])
            for j, d in enumerate(s.draws):
                d.texture = j
            return case["width"], case["height"], s.mvp, s.draws
        with ThreadPoolExecutor(4) as ex:
            return list(ex.map(one, range(case["views"])))
    d, mvp = _inside_scene(seed, case["tris"], case["width"], case["height"])
    return [(case["width"], case["height"], mvp, [d])]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "texture":
        return {"kind": kind, "ctx": sr.RenderContext(), "width": case["width"], "height": case["height"],
                "image": _noise(seed, case["width"], case["height"])}
    views = _views(case, seed)
    order = {"mixed": sr.ORDER_TRICOUNT, "clustered": sr.ORDER_TRICOUNT}.get(kind, case.get("order", 0))
    graph = case.get("graph", kind in ("mixed", "clustered"))
    ctx = sr.RenderContext(flags=sr.CFG_GRAPH if graph else 0, tile_order=order, wg_per_tile=case.get("parts", 0))
    shader = case.get("shader", "unlit")
    if shader == "sponza":
        ctx.set_sponza_constants(scenes.sponza_constants(seed & 0xFFFF, near=True))
    ntex = 1 + max(d.texture for v in views for d in v[3])
    size = case.get("tex", 256)
    texs = [ctx.CreateTexture(_noise(seed + 101 * k, size, size), size, size, True) for k in range(ntex)]
    fbs, calls = [], []
    for w, h, mvp, draws in views:
        fb = sr.FrameBuffer(ctx, w, h)
        fbs.append(fb)
        calls += [_call(fb, d, mvp, shader, texs[d.texture]) for d in draws]
    state = {"kind": kind, "ctx": ctx, "fbs": fbs, "texs": texs, "draws": ctx.PrepareDrawList(calls),
             "clears": ctx.PrepareClearList(fbs)}
    if kind != "inside":
        state["out"] = [_host((fb.m_height, fb.m_width), case.get("pinned", True)) for fb in fbs]
    return state


def run(state):
    ctx, kind = state["ctx"], state["kind"]
    if kind == "texture":
        tex = ctx.CreateTexture(state["image"], state["width"], state["height"], True)
        texels = tex.read().m_texels
        tex.release()
        return texels
    ctx.BeginFrame()
    ctx.ClearFrameBuffers(state["clears"], 0x20)
    ctx.DrawIndexedList(state["draws"])
    if kind == "inside":
        ctx.EndFrame(noalloc=True)
        colour, depth = state["fbs"][0].read_tiles()
        return colour.view(np.int32), depth.view(np.int32)
    ctx.EndFrame()
    if kind == "present":  # the previous frame has been shown before this one takes its place
        fb = state["fbs"][0]
        ctx.BlitWait(fb)
        return ctx.BlitAsync(fb, state["out"][0], bgra=True)
    for fb, out in zip(state["fbs"], state["out"]):
        ctx.Blit(fb, out)
    return state["out"]


# ---- what a pass cannot do without ----

def work(case):
    """Bytes: indices and vertices read once, the texels of a whole level-0 footprint of the picture at most, the image
    written once. Operations: about 150 per triangle (three transforms, edge and plane set-up) and 100 per pixel
    (interpolation, one bilinear sample)."""
    kind = case["kind"]
    if kind == "texture":
        n = case["width"] * case["height"]
        return {"bytes": 4.0 * n + 4.0 * n * 4 / 3, "flops": 64.0 * n}
    if kind == "mixed":  # the distribution's means: 80 k triangles, 0.8 megapixels a view
        views, tris, px, verts, shared = case["views"], 80000, 795000, 100000, False
    else:
        views, px = case.get("views", 1), case["width"] * case["height"]
        shared = kind in ("spheres", "cubes", "present")
        if kind == "cubes":
            tris, verts = 12 * case["grid"] ** 2, 24 * case["grid"] ** 2
        elif kind in ("spheres", "present"):
            tris, verts = 250 * case["spheres"], 182 * case["spheres"]
        else:
            tris, verts = case["tris"], 3 * case["tris"]
    read = (12.0 * tris + 32.0 * verts) * (1 if shared else views)
    out = 8.0 if kind == "inside" else 4.0
    lights = 16 * 25 if case.get("shader") == "sponza" else 0
    return {"bytes": read + views * px * out, "flops": views * (150.0 * tris + (100.0 + lights) * px)}


def exact(case, seed):
    """Every output is whole numbers, held equal: there is nothing to compare in 64 bits."""
    return None
