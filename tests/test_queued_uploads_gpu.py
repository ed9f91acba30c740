"""Uploads queued on the stream (batch tables, the backward pass's draw
tables) keep their order: a table changed while the work that reads it is
still queued, and batches larger than the staging they go through."""
import numpy as np
import pytest

from softlight_amd import api as A
from softlight_amd import scenes
from tests.parity import assert_parity, render_both

pytestmark = pytest.mark.gpu


def test_backward_tables_changed_while_queued(gpu_lib):
    """Backward passes of four framebuffers into one gradient buffer, then,
    with nothing waited for, into another: each gets its own sums."""
    ctx = A.SLContext(gpu_lib)
    sc = scenes.DiffScene(ctx, level=3, views=8, size=64, views_per_fbo=2, tex_size=32)
    sc.make_targets()
    sc.forward()
    sc.loss_grad_images()
    ctx.finish()
    other = ctx.create_vbo(np.zeros((sc.n_vertices, 4), dtype=np.float32))
    ctx.gradients_zero()
    for rep in range(3):
        for buf in (sc.grad_vbo, other):
            ctx.vbo_attach_gradient(sc.vbo, buf)
            for t in sc.targets:
                ctx.backward(t["fbo"], t["grad_image"])
    ctx.finish()
    a, b = (ctx.vbo_read(v, sc.n_vertices * 16, dtype=np.float32) for v in (sc.grad_vbo, other))
    assert float(np.abs(a).max()) > 0.0
    assert float(np.abs(a - b).max()) <= 1e-5 * float(np.abs(a).max())      # two orders of the same atomics


@pytest.mark.parametrize("meshes", [3, 150, 400])
def test_batches_around_the_staging_size(gpu_lib, oracle_lib, meshes):
    """The same batch drawn three times, with other uniforms in between."""
    def build(ctx):
        s = scenes.build_batched_scene(ctx, seed=4, n_meshes=meshes, median_tris=20, W=160, H=90, tex_size=32,
                                       n_textures=2, debug=True)
        s.render()
        u = A.sl_std_uniforms()
        for ubo in range(meshes):
            ctx.ubo_assign(ubo, np.float32([0.5, 0.25, 1.0, 1.0]), offset=A.sl_std_uniforms.tint.offset)
        s.render()
        ctx.finish()
        ctx.reset_stats()
        return s
    g, o = render_both(gpu_lib, oracle_lib, build)
    assert_parity(g, o)
