"""The smoothing passes' blocks (32x8 pixels and their halo) at the sizes
where they can go wrong, against the oracle: framebuffers of one block, one
pixel past it and ragged, with winners clipped by the frustum bounding some
pixels of a block (left to launches of their own) and not others, and more
draws than are searched in LDS.  Tolerances as the suite's batched smoothing check: 1e-5 for
images, 1e-4 of the largest for gradients."""
import numpy as np
import pytest

from softlight_amd import api as A
from softlight_amd import scenes

pytestmark = pytest.mark.gpu


def _run(lib, sigma, kw):
    ctx = A.SLContext(lib)
    sc = scenes.SmoothScene(ctx, **kw)
    sc.make_targets(sigma)
    sc.forward(sigma)
    sc.backward(sigma)
    ctx.finish()
    images, grads = [], [ctx.vbo_read(g, sc.pos[m].shape[0] * 16, dtype=np.float32) for m, g in enumerate(sc.grad_vbos)]
    for t in sc.targets:
        images += [ctx.texture_read(t["smooth"]), ctx.texture_read(t["grad_image"])]
        grads.append(ctx.vbo_read(t["pos_grad"], len(t["views"]) * len(sc.meshes) * sc.n_vertices_max * 8, dtype=np.float32))
    return images, grads


@pytest.mark.parametrize("distance", [4.0, 1.3])      # the nearer camera stands between the spheres: some are clipped
@pytest.mark.parametrize("kw", [
    dict(meshes=3, views=1, size=8, views_per_fbo=1),
    dict(meshes=3, views=1, size=32, views_per_fbo=1),
    dict(meshes=4, views=2, size=33, views_per_fbo=1),
    dict(meshes=8, views=9, size=41, views_per_fbo=9),
    dict(meshes=4, views=4, size=100, views_per_fbo=4),
])
def test_blocks_match_oracle(gpu_lib, oracle_lib, kw, distance):
    kw = dict(kw, min_tris=60, max_tris=400, tex_size=16, distance=distance)
    (gi, gg), (oi, og) = _run(gpu_lib, 0.05, kw), _run(oracle_lib, 0.05, kw)
    for a, b in zip(gi, oi):
        assert float(np.abs(a - b).max()) <= 1e-5 * max(1.0, float(np.abs(b).max()))
    assert any(float(np.abs(b).max()) > 0.0 for b in og)
    for a, b in zip(gg, og):
        assert float(np.abs(a - b).max()) <= 1e-4 * float(np.abs(b).max())
