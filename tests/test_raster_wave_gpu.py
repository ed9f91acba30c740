"""The raster of filled-triangle batches (one wave per 8x8 pixel block) at the
sizes where it can go wrong, against the CPU oracle bit for bit (depth,
per-pixel order and counts; colour within 1 LSB):

  targets      smaller than a block, one pixel past it, ragged in both axes,
               and wide: a fragment's barycentrics are stepped from its span's
               first pixel, thousands of columns away at most, at the cost of
               the steps and no more
  lists        63, 64, 65 and 129 records in a tile (64 are taken at a time)
  queue        more than 64 waiting fragments of one record and of one pixel
  depth        the seven functions mixed in one batch, with depth-raising draws
               between LESS draws, into float and half depth, and with blending
  small        batches on both sides of a triangle per 40 pixels, whose small
               records queue their own fragments
"""
import numpy as np
import pytest

from softlight_amd import api as A
from softlight_amd import scenes
from tests.parity import assert_parity, render_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(1, 1), (7, 5), (8, 8), (9, 8), (8, 9), (33, 17), (64, 64), (1500, 20)])
@pytest.mark.parametrize("blend", [A.SL_BLEND_OFF, A.SL_BLEND_ALPHA])
def test_target_sizes(gpu_lib, oracle_lib, size, blend):
    g, o = render_both(gpu_lib, oracle_lib, scenes.build_random_triangles, seed=21, ntri=150, W=size[0], H=size[1],
                       debug=True, blend=blend)
    assert_parity(g, o)


def _layers(ctx, W, H, n=8, debug=False, blend=A.SL_BLEND_OFF):
    """n pairs of triangles that cover the whole target, back to front: every
    fragment passes."""
    quad = np.float32([[-1, -1], [1, -1], [-1, 1], [-1, 1], [1, -1], [1, 1]])
    xyz = np.empty((n, 6, 3), dtype=np.float32)
    xyz[:, :, :2] = quad
    xyz[:, :, 2] = np.linspace(0.8, -0.8, n, dtype=np.float32)[:, None]
    rec = np.zeros((6 * n, 16), dtype=np.uint8)
    rec[:, 0:12] = xyz.reshape(-1, 3).view(np.uint8).reshape(-1, 12)
    rec[:, 12:16] = scenes.uniform_u8(17, 24 * n, stream=3).reshape(-1, 4)
    return scenes.build_from_vertex_records(ctx, rec, W, H, debug, shader_kw=dict(blend=blend))


@pytest.mark.parametrize("size", [(1031, 40), (4100, 9), (20000, 9)])
@pytest.mark.parametrize("blend", [A.SL_BLEND_OFF, A.SL_BLEND_ALPHA])
def test_layers_over_wide_targets(gpu_lib, oracle_lib, size, blend):
    g, o = render_both(gpu_lib, oracle_lib, _layers, W=size[0], H=size[1], debug=True, blend=blend)
    assert_parity(g, o)


def test_wide_fragments_cost_their_steps(gpu_lib):
    """Eight layers over 2 M pixels: at 3,840 columns a fragment takes up to 960
    steps, at 480 up to 120.  That costs the raster about three times as much;
    a jump over the steps, which fragments past some distance once took, cost
    it 29 times as much."""
    ms = {}
    for W, H in ((480, 4320), (3840, 540)):
        ctx = A.SLContext(gpu_lib)
        s = _layers(ctx, W, H)
        s.render()
        ctx.finish()
        best = []
        for _ in range(5):
            ctx.reset_stats()
            s.render()
            ctx.finish()
            best.append(ctx.stats()["ms_raster"])
        ms[W] = min(best)
        ctx.close()
    assert ms[3840] < 9.0 * ms[480], ms


@pytest.mark.parametrize("n", [1, 63, 64, 65, 129])
@pytest.mark.parametrize("config", [0, 3, 10, 11])
def test_list_lengths(gpu_lib, oracle_lib, n, config):
    """n triangles that each cover the whole target, nearer and nearer: every
    one is in every tile's list, covers whole blocks and passes."""
    def build(ctx):
        ctx.set_raster_config(config)
        rec = np.zeros((3 * n, 16), dtype=np.uint8)
        xyz = np.empty((n, 3, 3), dtype=np.float32)
        xyz[:] = [[-1.0, -1.0, 0.0], [1.0, -1.0, 0.0], [-1.0, 1.0, 0.0]]
        xyz[1::2, :, :2] *= -1.0                       # both halves of the target
        xyz[:, :, 2] = np.linspace(0.9, -0.9, n, dtype=np.float32)[:, None]
        xyz[:, 1, 2] += 0.05                           # slanted in depth
        rec[:, 0:12] = xyz.reshape(-1, 3).view(np.uint8).reshape(3 * n, 12)
        rec[:, 12:16] = scenes.uniform_u8(5, 12 * n, stream=3).reshape(3 * n, 4)
        return scenes.build_from_vertex_records(ctx, rec, 70, 45, True)
    g, o = render_both(gpu_lib, oracle_lib, build)
    assert_parity(g, o)


@pytest.mark.parametrize("depth_type", [A.SL_COLOR_R_FLOAT, A.SL_COLOR_R_HALF])
@pytest.mark.parametrize("blend", [A.SL_BLEND_OFF, A.SL_BLEND_ADDITIVE])
def test_depth_functions_in_one_batch(gpu_lib, oracle_lib, depth_type, blend):
    """Twelve draws of 60 triangles, each of another depth function and mask:
    LESS draws after GREATER, NOT_EQUAL and test-off draws see raised depths."""
    def build(ctx):
        s = scenes.build_from_vertex_records(ctx, scenes.random_triangle_vertices(31, 720), 93, 61, True,
                                             depth_type=depth_type)
        vao = s.draws[0][1].vaoId
        s.draws = []
        tests = [A.SL_DEPTH_TEST_LESS_THAN, A.SL_DEPTH_TEST_GREATER_THAN, A.SL_DEPTH_TEST_LESS_EQUAL,
                 A.SL_DEPTH_TEST_OFF, A.SL_DEPTH_TEST_LESS_THAN, A.SL_DEPTH_TEST_NOT_EQUAL,
                 A.SL_DEPTH_TEST_LESS_THAN, A.SL_DEPTH_TEST_GREATER_EQUAL, A.SL_DEPTH_TEST_EQUAL,
                 A.SL_DEPTH_TEST_LESS_THAN, A.SL_DEPTH_TEST_OFF, A.SL_DEPTH_TEST_LESS_EQUAL]
        for k, t in enumerate(tests):
            sh = scenes.gouraud_shader(ctx, depth_test=t, blend=blend if k % 3 == 1 else A.SL_BLEND_OFF,
                                       depth_mask=A.SL_DEPTH_MASK_OFF if k == 4 else A.SL_DEPTH_MASK_ON)
            s.draws.append(("draw_shader", A.sl_mesh(vao, 180 * k, 180 * (k + 1), A.RENDER_MODE_TRIANGLES, 0), sh))
        return s
    g, o = render_both(gpu_lib, oracle_lib, build)
    assert_parity(g, o)


@pytest.mark.parametrize("mode", [A.RENDER_MODE_TRI_WIRE, A.RENDER_MODE_LINES, A.RENDER_MODE_POINTS])
@pytest.mark.parametrize("size", [(1, 1), (7, 9), (8, 8), (33, 17), (70, 45)])
@pytest.mark.parametrize("blend,depth_type", [(A.SL_BLEND_OFF, A.SL_COLOR_R_FLOAT), (A.SL_BLEND_ALPHA, A.SL_COLOR_R_HALF)])
def test_render_modes_target_sizes(gpu_lib, oracle_lib, mode, size, blend, depth_type):
    """Wireframe, lines (some of no length) and points on targets around a
    block's size; the opaque batches with heavy tiles split into parts of 3."""
    def build(ctx):
        ctx.set_raster_split(3)
        rec = scenes.random_triangle_vertices(41, 80).copy()
        rec[6:12] = rec[0:6]                                # repeated primitives: equal depths
        rec[13] = rec[12]                                   # a line of no length
        rec[60:90, 0:8] = rec[60, 0:8]                      # a pile on one texel
        return scenes.build_from_vertex_records(ctx, rec, size[0], size[1], True, mode=mode, depth_type=depth_type,
                                                shader_kw=dict(blend=blend))
    g, o = render_both(gpu_lib, oracle_lib, build)
    assert_parity(g, o)


@pytest.mark.parametrize("tiles", [(4, 4), (17, 1), (1, 17), (20, 7)])
def test_bin_entries_of_large_records(gpu_lib, oracle_lib, tiles):
    """Triangles of up to 16 tiles (whose entries the emitting lane writes),
    just above (written by a wave) and of many tiles, among small ones, with
    parts of them clipped; 32x16 tiles."""
    def build(ctx):
        W, H = 32 * 24, 16 * 20
        rec = scenes.random_triangle_vertices(51, 700).copy()
        xyz = rec[:, 0:12].copy().view(np.float32).reshape(-1, 3, 3)
        k = np.arange(xyz.shape[0])
        sx, sy = 2.0 * 32 * tiles[0] / W, 2.0 * 16 * tiles[1] / H
        size = np.where((k % 3 == 0)[:, None, None], np.float32([sx, sy, 1.0]), np.float32([0.02, 0.03, 1.0]))
        xyz[:, 1:] = xyz[:, :1] + (xyz[:, 1:] * size).astype(np.float32)
        rec[:, 0:12] = xyz.astype(np.float32).reshape(-1, 3).view(np.uint8).reshape(-1, 12)
        return scenes.build_from_vertex_records(ctx, rec, W, H, True)
    g, o = render_both(gpu_lib, oracle_lib, build)
    assert_parity(g, o)


@pytest.mark.parametrize("size,n", [((40, 10), 9), ((40, 10), 10), ((9, 7), 700), ((200, 40), 260), ((130, 70), 3000)])
@pytest.mark.parametrize("debug", [False, True])
@pytest.mark.parametrize("depth_type", [A.SL_COLOR_R_FLOAT, A.SL_COLOR_R_HALF])
def test_small_triangles(gpu_lib, oracle_lib, size, n, debug, depth_type):
    """Triangles of a pixel or three, every seventh over many columns and a run
    of them piled on one pixel, opaque and blended draws in turn and one draw
    that raises depths: batches of at least a triangle per 40 pixels (the
    first case is just below) take the instances whose small records queue
    their own fragments, lists with wide or raising records the wave's steps."""
    def build(ctx):
        rec = scenes.random_triangle_vertices(61, n).copy()
        xyz = rec[:, 0:12].copy().view(np.float32).reshape(-1, 3, 3)
        k = np.arange(n)
        px = np.float32([2.0 / size[0], 2.0 / size[1], 1.0])
        ext = np.where((k % 7 == 0)[:, None, None], np.float32([0.9, 0.1, 1.0]), 6.0 * px).astype(np.float32)
        xyz[:, 1:] = xyz[:, :1] + xyz[:, 1:] * ext
        xyz[n // 3:n // 2, :, :2] = xyz[n // 3, :, :2]          # a pile
        if n >= 700:
            xyz[k % 7 == 0, 1:] = xyz[k % 7 == 0, :1]           # and lists of small ones only
            xyz[: n // 4: 7] = xyz[n // 4]
        rec[:, 0:12] = xyz.astype(np.float32).reshape(-1, 3).view(np.uint8).reshape(-1, 12)
        s = scenes.build_from_vertex_records(ctx, rec, size[0], size[1], debug, depth_type=depth_type)
        vao = s.draws[0][1].vaoId
        s.draws = []
        step = 3 * (n // 6)
        for d, (blend, test) in enumerate([(A.SL_BLEND_OFF, A.SL_DEPTH_TEST_LESS_THAN), (A.SL_BLEND_ALPHA, A.SL_DEPTH_TEST_LESS_EQUAL),
                                           (A.SL_BLEND_OFF, A.SL_DEPTH_TEST_LESS_EQUAL), (A.SL_BLEND_ADDITIVE, A.SL_DEPTH_TEST_GREATER_THAN),
                                           (A.SL_BLEND_ALPHA, A.SL_DEPTH_TEST_LESS_THAN), (A.SL_BLEND_OFF, A.SL_DEPTH_TEST_EQUAL)]):
            sh = scenes.gouraud_shader(ctx, depth_test=test, blend=blend)
            end = 3 * n if d == 5 else step * (d + 1)
            s.draws.append(("draw_shader", A.sl_mesh(vao, step * d, end, A.RENDER_MODE_TRIANGLES, 0), sh))
        return s
    g, o = render_both(gpu_lib, oracle_lib, build)
    assert_parity(g, o)
