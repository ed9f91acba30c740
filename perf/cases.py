"""What the draw path is measured on: the calls that a program makes with it.

Every case is one pass of such a program through the public binding
(`softlight_amd.api`): record the clears and draws, let the frame run, and
read what the program uses.  A renderer reads the finished image (depth and
the G-buffer too, where it asks for them) into page-locked memory that it
keeps; an optimiser runs the forward and backward passes and reads the
gradients.  Sizes and distributions are those of the repository's scenes
(random clip-space triangles, instanced UV spheres, batched meshes, many
views of an icosphere, smoothed coverage) and of its benchmark and tests.

The kinds, and the ranges that `draw` spreads them over:

  triangles  64 .. 4,096 random triangles (or up to 20,000 points or lines)
             into 96x64 .. 1280x720, each colour and depth format, blending
  spheres    1 .. 64 instances of a textured UV sphere of 12^2 .. 256^2
             segments at 160x120 .. 1920x1080, filled, wireframe, lines,
             points, or with the four outputs of a G-buffer
  meshes     4 .. 1,000 meshes of uneven sizes, a draw call each, a fifth of
             them blended; recorded every frame or replayed as a captured
             frame; read as drawn or blitted to a window's back-buffer
  views      2 .. 32 views of a coloured and textured icosphere, forward,
             L2 loss and backward, 64^2 .. 512^2 pixels a view
  smooth     2 .. 16 views of several meshes with smoothed coverage, forward
             and backward to colours, texels and screen positions
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import softlight_amd
from softlight_amd import api as A
from softlight_amd import scenes

_COLOR = {"rgba8": A.SL_COLOR_RGBA_8U, "rgb8": A.SL_COLOR_RGB_8U, "rgba32f": A.SL_COLOR_RGBA_FLOAT,
          "rgb565": A.SL_COLOR_RGB_565}
_DEPTH = {"r32f": A.SL_COLOR_R_FLOAT, "r16f": A.SL_COLOR_R_HALF}
_BLEND = {"off": A.SL_BLEND_OFF, "alpha": A.SL_BLEND_ALPHA, "additive": A.SL_BLEND_ADDITIVE}
_MODE = {"fill": A.RENDER_MODE_TRIANGLES, "wire": A.RENDER_MODE_TRI_WIRE, "lines": A.RENDER_MODE_LINES,
         "points": A.RENDER_MODE_POINTS}
# bytes a texel, and the type and components that a program reads it as
_TEXEL = {"rgba8": (4, torch.uint8, 4), "rgb8": (3, torch.uint8, 3), "rgba32f": (16, torch.float32, 4),
          "rgb565": (2, torch.int16, 1), "r32f": (4, torch.float32, 1), "r16f": (2, torch.float16, 1)}


def listed():
    return [
        # the smallest call: a few hundred triangles into a thumbnail; launches and round trips
        dict(name="triangles_256_128x96", kind="triangles", n=256, W=128, H=96, mode="fill", color="rgba8",
             depth="r32f", blend="off", read_depth=True),
        # large overlapping triangles at the benchmark's size, the library's default knobs; colour and depth used
        dict(name="triangles_4096_640x480", kind="triangles", n=4096, W=640, H=480, mode="fill", color="rgba8",
             depth="r32f", blend="off", read_depth=True),
        # blended large triangles into a float target of a ragged size
        dict(name="triangles_blend_801x603", kind="triangles", n=1200, W=801, H=603, mode="fill", color="rgba32f",
             depth="r32f", blend="alpha", read_depth=False),
        # an interactive scene in the reference demos' target formats (RGB8 + half depth)
        dict(name="spheres_8x64_640x480_rgb8", kind="spheres", instances=8, segments=64, W=640, H=480, tex=256,
             mode="fill", color="rgb8", depth="r16f", read_depth=False, config=-1, wg_per_cu=0),
        # the benchmark's frame: 8.4 M triangles at 1080p, with its tuned tile
        dict(name="spheres_64x256_1080p", kind="spheres", instances=64, segments=256, W=1920, H=1080, tex=1024,
             mode="fill", color="rgba8", depth="r32f", read_depth=False, config=5, wg_per_cu=8),
        # lines of a mesh (a debug view): many tiny primitives, uneven tiles
        dict(name="spheres_lines_1280x720", kind="spheres", instances=16, segments=128, W=1280, H=720, tex=256,
             mode="lines", color="rgba8", depth="r32f", read_depth=False, config=-1, wg_per_cu=0),
        # a deferred renderer's G-buffer: four colour attachments and depth
        dict(name="spheres_gbuffer_1280x720", kind="spheres", instances=16, segments=96, W=1280, H=720, tex=512,
             mode="gbuffer", color="rgba8", depth="r32f", read_depth=True, config=-1, wg_per_cu=0),
        # a small scene recorded every frame, presented into a window of another size
        dict(name="meshes_60_present_1000x750", kind="meshes", meshes=60, median=800, W=1000, H=750, captured=False,
             present=True, config=-1, split=-1),
        # the batched frame: 1000 meshes at 1080p as a captured frame, with its tuned tile and bin capacity
        dict(name="meshes_1000_1080p", kind="meshes", meshes=1000, median=2000, W=1920, H=1080, captured=True,
             present=False, config=3, split=1024),
        # a small optimisation step: four thumbnails of a coarse mesh
        dict(name="views_4x128", kind="views", views=4, size=128, level=3, per=4, tex=128),
        # the benchmark's optimisation step: 32 views of 20,480 triangles
        dict(name="views_32x512", kind="views", views=32, size=512, level=5, per=8, tex=512),
        # smoothed coverage, forward and backward: 16 of the benchmark's views of its eight meshes
        dict(name="smooth_16x512", kind="smooth", views=16, size=512, meshes=8, min_tris=5000, max_tris=60000, per=8,
             tex=512, sigma=0.01),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi, aspect=(1.2, 1.8)):
    W = _log(rng, lo, hi)
    return W, max(8, int(round(W / rng.uniform(*aspect))))


def draw(rng):
    kind = rng.choice(["triangles", "triangles", "spheres", "spheres", "meshes", "views", "smooth"])
    if kind == "triangles":
        mode = rng.choice(["fill", "fill", "fill", "wire", "lines", "points"])
        W, H = _size(rng, 96, 1280)
        n = _log(rng, 64, 4096 if mode in ("fill", "wire") else 20000)
        if mode in ("fill", "wire"):      # no longer lists in a tile, and no more covered pixels, than the listed frame
            n = max(64, min(n, int(4096 * W / 640), int(4096 * 640 * 480 / (W * H))))
        color = rng.choice(["rgba8", "rgba8", "rgb8", "rgba32f", "rgb565"])
        return dict(kind=kind, n=n, W=W, H=H, mode=mode, color=color,
                    depth=rng.choice(["r32f", "r32f", "r16f"]), blend=rng.choice(["off", "off", "alpha", "additive"]),
                    read_depth=rng.random() < 0.5)
    if kind == "spheres":
        mode = rng.choice(["fill", "fill", "fill", "wire", "lines", "points", "gbuffer"])
        W, H = _size(rng, 160, 1920)
        segments = _log(rng, 12, 256)
        instances = _log(rng, 1, 64)
        if mode in ("lines", "points"):   # no more primitives than the listed lines
            instances = max(1, min(instances, int(16 * 128 * 128 / (segments * segments))))
        return dict(kind=kind, instances=instances, segments=segments, W=W, H=min(H, 1080), tex=_log(rng, 32, 1024),
                    mode=mode, color=rng.choice(["rgba8", "rgba8", "rgb8"]) if mode != "gbuffer" else "rgba8",
                    depth=rng.choice(["r32f", "r32f", "r16f"]), read_depth=rng.random() < 0.3,
                    config=rng.choice([-1, -1, -1, 3, 5]), wg_per_cu=rng.choice([0, 0, 8]))
    if kind == "meshes":
        W, H = _size(rng, 320, 1920)
        meshes = _log(rng, 4, 1000)
        return dict(kind=kind, meshes=meshes, median=_log(rng, 100, 2000), W=W, H=min(H, 1080),
                    captured=meshes > 200 or rng.random() < 0.5, present=rng.random() < 0.4,
                    config=rng.choice([-1, -1, 3]), split=rng.choice([-1, -1, 1024]))
    if kind == "views":
        return dict(kind=kind, views=_log(rng, 2, 32), size=_log(rng, 64, 512), level=rng.choice([2, 3, 4, 5]),
                    per=rng.choice([1, 2, 4, 8]), tex=_log(rng, 32, 512))
    return dict(kind=kind, views=_log(rng, 2, 16), size=_log(rng, 64, 512), meshes=rng.choice([1, 2, 4, 8]),
                min_tris=_log(rng, 200, 5000), max_tris=_log(rng, 6000, 60000), per=rng.choice([2, 4, 8]),
                tex=_log(rng, 32, 512), sigma=rng.choice([0.01, 0.03, 0.1]))


class _Readback:
    """Textures and vertex buffers that the program reads after each pass,
    each into page-locked memory of its own that it keeps."""

    def __init__(self, ctx):
        self.ctx, self.items = ctx, []

    def texture(self, name, tex, fmt, w, h):
        bpt, dtype, comps = _TEXEL[fmt]
        host = torch.empty((h, w, comps), dtype=dtype, pin_memory=True)
        self.items.append((name, self.ctx.lib.texture_read, tex, host, (w * h * bpt,)))

    def buffer(self, name, vbo, shape):
        host = torch.empty(shape, dtype=torch.float32, pin_memory=True)
        self.items.append((name, self.ctx.lib.vbo_read, vbo, host, (0, host.numel() * 4)))

    def __call__(self):
        out = {}
        for name, fn, handle, host, args in self.items:
            rc = fn(self.ctx.h, handle, ctypes.c_void_p(host.data_ptr()), *args)
            if rc != A.SL_OK:
                raise RuntimeError("reading %s back failed (%d)" % (name, rc))
            out[name] = host
        return out


def _gbuffer_scene(ctx, case, seed):
    """The sphere scene with the four outputs of SL_PROGRAM_LAMBERT_MRT."""
    s = scenes.build_sphere_scene(ctx, seed=seed, n_instances=case["instances"], stacks=case["segments"],
                                  sectors=case["segments"], W=case["W"], H=case["H"], tex_size=case["tex"],
                                  depth_type=_DEPTH[case["depth"]])
    W, H = case["W"], case["H"]
    colors = [s.color] + [ctx.create_texture(_COLOR[case["color"]], W, H) for _ in range(3)]
    s.fbo = ctx.create_framebuffer(colors, s.depth)
    vs = A.sl_vertex_shader(3, A.SL_CULL_BACK_FACE, A.SL_PROGRAM_LAMBERT_MRT)
    fs = A.sl_fragment_shader(3, 4, A.SL_BLEND_OFF, A.SL_DEPTH_TEST_LESS_THAN, A.SL_DEPTH_MASK_ON,
                              A.SL_PROGRAM_LAMBERT_MRT)
    s.shader = ctx.create_shader(vs, fs, 0)        # the scene's one uniform buffer
    return s, colors


def prepare(case, seed):
    seed = int(seed) & 0x7FFFFFFF
    ctx = softlight_amd.new_context()
    read = _Readback(ctx)
    kind = case["kind"]
    if kind == "triangles":
        W, H = case["W"], case["H"]
        kw = dict(color_type=_COLOR[case["color"]], depth_type=_DEPTH[case["depth"]])
        if case["mode"] in ("fill", "wire"):
            s = scenes.build_random_triangles(ctx, seed, case["n"], W, H, wire=case["mode"] == "wire",
                                              blend=_BLEND[case["blend"]], **kw)
        else:
            per = 2 if case["mode"] == "lines" else 1
            rec = scenes.random_triangle_vertices(seed, -(-per * case["n"] // 3))[:per * case["n"]]
            s = scenes.build_from_vertex_records(ctx, np.ascontiguousarray(rec), W, H, mode=_MODE[case["mode"]],
                                                 shader_kw=dict(blend=_BLEND[case["blend"]]), **kw)
        read.texture("color", s.color, case["color"], W, H)
        if case["read_depth"]:
            read.texture("depth", s.depth, case["depth"], W, H)
        return dict(case=case, ctx=ctx, scene=s, read=read)
    if kind == "spheres":
        W, H = case["W"], case["H"]
        colors = []
        if case["mode"] == "gbuffer":
            s, colors = _gbuffer_scene(ctx, case, seed)
        else:
            s = scenes.build_sphere_scene(ctx, seed=seed, n_instances=case["instances"], stacks=case["segments"],
                                          sectors=case["segments"], W=W, H=H, tex_size=case["tex"],
                                          wire=case["mode"] == "wire",
                                          prim=case["mode"] if case["mode"] in ("lines", "points") else "triangles",
                                          color_type=_COLOR[case["color"]], depth_type=_DEPTH[case["depth"]])
        if case["config"] >= 0:
            ctx.set_raster_config(case["config"])
        if case["wg_per_cu"] > 0:
            ctx.set_raster_occupancy(case["wg_per_cu"])
        for k, tex in enumerate(colors or [s.color]):
            read.texture("color%d" % k, tex, case["color"], W, H)
        if case["read_depth"]:
            read.texture("depth", s.depth, case["depth"], W, H)
        return dict(case=case, ctx=ctx, scene=s, read=read, extra=range(1, len(colors)))
    if kind == "meshes":
        W, H = case["W"], case["H"]
        s = scenes.build_batched_scene(ctx, seed=seed, n_meshes=case["meshes"], median_tris=case["median"], W=W, H=H,
                                       max_tris=100 * case["median"])
        if case["config"] >= 0:
            ctx.set_raster_config(case["config"])
        if case["split"] >= 0:
            ctx.set_raster_split(case["split"])
        window = None
        if case["present"]:
            ww, wh = max(1, W * 4 // 5), max(1, H * 4 // 5)
            window = ctx.create_texture(A.SL_COLOR_RGBA_8U, ww, wh)
            read.texture("window", window, "rgba8", ww, wh)
        else:
            read.texture("color", s.color, "rgba8", W, H)
        if case["captured"]:
            s.render()
            ctx.frame_graph_capture()
        return dict(case=case, ctx=ctx, scene=s, read=read, window=window)
    if kind == "views":
        sc = scenes.DiffScene(ctx, seed=seed, level=case["level"], views=case["views"], size=case["size"],
                              views_per_fbo=case["per"], tex_size=case["tex"])
        sc.make_targets()
        read.buffer("grad_colors", sc.grad_vbo, (sc.n_vertices, 4))
        read.texture("grad_texels", sc.grad_tex, "rgba32f", case["tex"], case["tex"])
        return dict(case=case, ctx=ctx, scene=sc, read=read)
    # the meshes' sizes and the cameras belong to the case, so that the gradient
    # buffers have one shape; orientations, colours and texels to the seed
    sc = scenes.SmoothScene(ctx, seed=6, meshes=case["meshes"], min_tris=case["min_tris"],
                            max_tris=case["max_tris"], views=case["views"], size=case["size"],
                            views_per_fbo=case["per"], tex_size=case["tex"])
    turns = scenes.uniform(seed, 4 * case["meshes"], -1.0, 1.0, stream=50).astype(np.float64).reshape(-1, 4)
    for m, v in enumerate(sc.pos):
        R = scenes.rotation(turns[m, :3] + (0.0, 0.0, 1e-3), math.pi * turns[m, 3])
        v[:, 0:3] = (v[:, 0:3].astype(np.float64) @ R.T).astype(np.float32)
        v[:, 3:6] = scenes.uniform01(seed + m, v.shape[0] * 3, stream=51).reshape(-1, 3)
        ctx.vbo_assign(sc.vbos[m], v)
    texels = scenes.uniform01(seed, case["tex"] ** 2 * 4, stream=52).reshape(case["tex"], case["tex"], 4)
    ctx.texture_set_texels(sc.tex, texels)
    sc.make_targets(case["sigma"])
    for m, g in enumerate(sc.grad_vbos):
        read.buffer("grad_colors%d" % m, g, (sc.pos[m].shape[0], 4))
    read.texture("grad_texels", sc.grad_tex, "rgba32f", case["tex"], case["tex"])
    for k, t in enumerate(sc.targets):
        read.buffer("grad_positions%d" % k, t["pos_grad"], (len(t["views"]) * case["meshes"], sc.n_vertices_max, 2))
    return dict(case=case, ctx=ctx, scene=sc, read=read)


def run(state):
    case, ctx, s = state["case"], state["ctx"], state["scene"]
    kind = case["kind"]
    if kind == "views":
        s.forward()
        s.loss_grad_images()
        s.backward()
    elif kind == "smooth":
        s.forward(case["sigma"])
        s.backward(case["sigma"])
    elif kind == "meshes":
        if case["captured"]:
            ctx.frame_graph_launch()
        else:
            s.render()
        if state["window"] is not None:
            ctx.blit(state["window"], s.color)
    else:
        for k in state.get("extra", ()):
            ctx.clear_color_buffer(s.fbo, k, (0.0, 0.0, 0.0, 0.0))
        s.render()
    return state["read"]()


def _image_bytes(case):
    return case["W"] * case["H"] * (_TEXEL[case["color"]][0] + (_TEXEL[case["depth"]][0]))


def work(case):
    """The inputs once, the targets (and gradients) once; the vertex program
    and the samples that a frame of the kind covers on average."""
    kind = case["kind"]
    if kind == "triangles":
        verts = case["n"] * {"fill": 3, "wire": 3, "lines": 2, "points": 1}[case["mode"]]
        # a random clip-space triangle covers about 1/13 of the screen
        covered = {"fill": case["W"] * case["H"] / 13, "wire": 2 * (case["W"] + case["H"]),
                   "lines": (case["W"] + case["H"]) / 2, "points": 1}[case["mode"]] * case["n"]
        return dict(bytes=16 * verts + _image_bytes(case), flops=30 * verts + 8 * covered)
    if kind == "spheres":
        n = case["segments"]
        verts, idx = (n + 1) ** 2, 6 * n * (n - 1)
        image = _image_bytes(case) + (3 * 4 * case["W"] * case["H"] if case["mode"] == "gbuffer" else 0)
        return dict(bytes=32 * verts + 4 * idx + 64 * case["instances"] + 4 * case["tex"] ** 2 + image,
                    flops=case["instances"] * verts * 80 + case["W"] * case["H"] * 30)
    if kind == "meshes":
        tris = case["meshes"] * case["median"] * 1.65          # the log-normal's mean over its median
        image = 8 * case["W"] * case["H"] * (1.32 if case["present"] else 1.0)
        return dict(bytes=tris * (12 + 16) + 16 * 4 * 512 ** 2 + 1024 * case["meshes"] + image,
                    flops=tris * 0.5 * 80 + case["W"] * case["H"] * 60)
    pixels = case["views"] * case["size"] ** 2
    params = 2 * 16 * case["tex"] ** 2
    if kind == "views":
        verts, tris = 10 * 4 ** case["level"] + 2, 20 * 4 ** case["level"]
        # colour, depth and visibility written, the target read; gradients written
        return dict(bytes=verts * (32 + 16) + 12 * tris + params + pixels * (16 + 4 + 16 + 16),
                    flops=case["views"] * verts * 80 + pixels * 100)
    tris = case["meshes"] * (case["max_tris"] - case["min_tris"]) / math.log(case["max_tris"] / case["min_tris"])
    # as above, and the smoothed image and its adjoint written; a float2 per view, mesh and vertex
    return dict(bytes=tris * (0.5 * (32 + 16) + 12) + params + pixels * (16 + 4 + 16 + 16 + 16 + 16) +
                case["views"] * tris * 0.5 * 8, flops=case["views"] * tris * 0.5 * 80 + pixels * 200)


def exact(case, seed):
    """No case has a 64-bit counterpart.  Images and depth are defined by the
    draw path's own float32 decisions (span ends, depth ties, submission
    order), and the gradients sum over the pixels' winners: in 64 bits some
    pixels have another winner, and the result is that of another image."""
    return None
