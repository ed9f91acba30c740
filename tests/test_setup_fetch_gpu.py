"""Vertex and index fetches of one load each, and the block sums of the counting
pass's chunks, against the CPU oracle bit for bit:

  attributes  1 to 4 floats each, at odd dword offsets, the last vertex ending
              with its buffer, with ids past it (zeros)
  indices     8, 16 and 32 bits, the last triangle reaching past the buffer
              (index 0)
  instances   one (no division) and several
  chunks      one block of 1,024 chunks of 256 triangles, and a chunk more
"""
import numpy as np
import pytest

from softlight_amd import api as A
from softlight_amd import scenes
from tests.parity import assert_parity, render_both

pytestmark = pytest.mark.gpu

DIMS = [A.VERTEX_DIMENSION_1, A.VERTEX_DIMENSION_2, A.VERTEX_DIMENSION_3, A.VERTEX_DIMENSION_4]


@pytest.mark.parametrize("pos,col", [(2, 1), (3, 2), (3, 3), (4, 4), (3, 4)])
@pytest.mark.parametrize("index", [None, np.uint8, np.uint16, np.uint32])
def test_attribute_and_index_widths(gpu_lib, oracle_lib, pos, col, index):
    def build(ctx):
        n = 150
        w = 1 + pos + col                                     # a leading dword: offsets 4 and 4 + 4 pos
        rec = np.zeros((n, w), dtype=np.float32)
        rec[:, 1:1 + pos] = scenes.uniform(71, n * pos, -1.0, 1.0, stream=1).reshape(n, pos)
        if pos == 4:
            rec[:, 4] = 1.0 + 0.5 * np.abs(rec[:, 4])
        rec[:, 1 + pos:] = scenes.uniform(71, n * col, 0.0, 1.0, stream=2).reshape(n, col)
        s = scenes.build_from_vertex_records(ctx, scenes.random_triangle_vertices(1, 1), 65, 47, True)
        ibo = None
        end = n
        if index is not None:
            ids = (scenes.uniform_u8(71, 298, stream=3).astype(np.int64) % (n + 3)).astype(index)   # some past the buffer
            ibo = ctx.create_ibo(ids)
            end = 300                                         # two elements past the index buffer
        vao = ctx.create_vao(ctx.create_vbo(rec), ibo, [(4, 4 * w, DIMS[pos - 1], A.VERTEX_DATA_FLOAT),
                                                        (4 + 4 * pos, 4 * w, DIMS[col - 1], A.VERTEX_DATA_FLOAT)])
        mode = A.RENDER_MODE_INDEXED_TRIANGLES if index is not None else A.RENDER_MODE_TRIANGLES
        s.draws = [("draw", A.sl_mesh(vao, 0, end, mode, 0), inst) for inst in (1, 3)]
        return s
    g, o = render_both(gpu_lib, oracle_lib, build)
    assert_parity(g, o)


@pytest.mark.parametrize("ntri", [256 * 1024, 256 * 1024 + 1])
def test_chunk_blocks(gpu_lib, oracle_lib, ntri):
    def build(ctx):
        rec = scenes.random_triangle_vertices(73, ntri).copy()
        xyz = rec[:, 0:12].copy().view(np.float32).reshape(-1, 3, 3)
        xyz[:, 1:] = xyz[:, :1] + xyz[:, 1:] * np.float32(0.03)
        rec[:, 0:12] = xyz.astype(np.float32).reshape(-1, 3).view(np.uint8).reshape(-1, 12)
        return scenes.build_from_vertex_records(ctx, rec, 320, 200, True)
    g, o = render_both(gpu_lib, oracle_lib, build)
    assert_parity(g, o)


@pytest.mark.parametrize("tiles,n", [((1, 1), 1), ((1, 1), 65), ((1, 1), 257), ((2, 1), 64), ((3, 1), 63), ((8, 8), 5),
                                     ((13, 5), 16), ((24, 20), 300)])
def test_bin_entry_counts(gpu_lib, oracle_lib, tiles, n):
    """n triangles that each reach every one of the 8x8 tiles: a power of two of
    them and around it, entries below, at and past 64, a 256-entry block and
    512 such blocks (144,000 entries, where a block's length grows)."""
    def build(ctx):
        ctx.set_raster_config(10)                               # 8x8 tiles
        rec = scenes.random_triangle_vertices(79, n).copy()
        xyz = rec[:, 0:12].copy().view(np.float32).reshape(-1, 3, 3)
        xyz[:, :, :2] = [[-1.0, -1.0], [1.0, -1.0], [-1.0, 1.0]]
        xyz[1::2, :, :2] *= -1.0
        rec[:, 0:12] = xyz.reshape(-1, 3).view(np.uint8).reshape(-1, 12)
        return scenes.build_from_vertex_records(ctx, rec, 8 * tiles[0], 8 * tiles[1], True)
    g, o = render_both(gpu_lib, oracle_lib, build)
    assert_parity(g, o)
