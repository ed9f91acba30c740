"""The adjoint's workgroup aggregation (16x16 pixels) at the sizes where it can
go wrong, against the oracle's scalar adjoint (summed in double).  Tolerance:
1e-4 of the largest gradient, as the suite's other adjoint checks; a block's
sum of at most 1,024 float products and the few hundred blocks that add to one
destination round to well below it.

  targets    smaller than a block and ragged in both axes
  lists      a texture of 2x2 to 4x4 texels (hundreds of items a texel, long
             lists of a vertex), and one so fine that a block's taps outnumber
             the table's groups (items that go to memory directly)
  draws      more draws in a framebuffer than are searched in LDS, and several
             meshes (destination buffers) in a block
  nearest    one tap a pixel
"""
import numpy as np
import pytest

from softlight_amd import api as A
from softlight_amd import scenes

pytestmark = pytest.mark.gpu


def _gradients(lib, kw):
    sc = scenes.DiffScene(A.SLContext(lib), **kw)
    sc.make_targets()
    sc.forward()
    sc.loss_grad_images()
    sc.backward()
    return sc.gradients()


@pytest.mark.parametrize("kw", [
    dict(level=1, views=1, size=7, views_per_fbo=1, tex_size=8),
    dict(level=2, views=3, size=33, views_per_fbo=2, tex_size=16),
    dict(level=0, views=2, size=128, views_per_fbo=2, tex_size=2),
    dict(level=1, views=2, size=96, views_per_fbo=1, tex_size=4),
    dict(level=4, views=2, size=40, views_per_fbo=2, tex_size=1024),
    dict(level=2, views=70, size=16, views_per_fbo=70, tex_size=32),
    dict(level=3, views=2, size=50, views_per_fbo=2, tex_size=64, flags=A.SL_UNIFORM_SAMPLE_NEAREST),
])
def test_gradients_match_oracle(gpu_lib, oracle_lib, kw):
    for got, ref in zip(_gradients(gpu_lib, kw), _gradients(oracle_lib, kw)):
        assert float(np.abs(ref).max()) > 0.0
        assert float(np.abs(ref - got).max()) <= 1e-4 * float(np.abs(ref).max())


def test_several_meshes_in_a_block(gpu_lib, oracle_lib):
    """Eight overlapping spheres, each with a colour gradient of its own, in
    views of 48x48 pixels: most blocks hold several destination buffers (all
    eight meshes and the texture get gradients)."""
    outs = []
    for lib in (gpu_lib, oracle_lib):
        ctx = A.SLContext(lib)
        sc = scenes.SmoothScene(ctx, meshes=8, min_tris=100, max_tris=400, views=4, size=48, views_per_fbo=4, tex_size=32)
        sc.make_targets(0.0)
        sc.forward(0.0)
        sc.backward(0.0)
        ctx.finish()
        outs.append([ctx.vbo_read(g, sc.pos[m].shape[0] * 16, dtype=np.float32) for m, g in enumerate(sc.grad_vbos)] +
                    [ctx.texture_read(sc.grad_tex)])
    for got, ref in zip(*outs):
        assert float(np.abs(ref).max()) > 0.0
        assert float(np.abs(ref - got).max()) <= 1e-4 * float(np.abs(ref).max())
