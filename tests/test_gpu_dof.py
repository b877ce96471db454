"""Depth of field at the edges of its 64x32 tiles and of its halos: viewports
of one pixel, one short of a tile, a tile, one past it and several tiles, at
the origin and inside a larger surface, boxes below and from the radius that
reads prefix sums, and the largest radius of either halo; tap means against
integer division are part of tests/cpp/arith_check.cpp."""
import numpy as np
import pytest

import oracle
from swegl_amd import host, scenes
from swegl_amd.device import Context
from swegl_amd.host import Surface, pixel_shader_light_and_texture, viewport_t

from _helpers import compare, gpu_render

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("taps,rmax", [("box", 2), ("box", 3), ("box", 8), ("box", 9), ("box", 16), ("tap9", 0),
                                       ("tap9", 8), ("tap9", 16)])
@pytest.mark.parametrize("x,y,w,h", [(0, 0, 1, 1), (0, 0, 63, 31), (0, 0, 64, 32), (5, 3, 65, 33), (0, 0, 7, 100),
                                     (3, 9, 200, 97)])
def test_dof_tile_edges(ctx, taps, rmax, x, y, w, h):
    scene, vps = scenes.heightfield_scene(5, n=60, width=w, height=h, tex=64, dof=False)
    rng = np.random.default_rng(w * h)
    for t in scene.images:
        t.bitmap[...] = rng.integers(0, 1 << 32, t.bitmap.shape, np.uint32)
    vp = viewport_t(x, y, w, h, Surface(x + w + 2, y + h + 1), pixel_shader_light_and_texture(), 0)
    vp.m_camera = vps[0].m_camera
    vp.set_post_shader(host.post_shader_depth_box(2.0, 1.5, vp, max_radius=rmax, taps=taps))
    want = oracle.render(scene, [vp])[0]
    compare(gpu_render(ctx, scene, [vp])[0], want, colour_tol=2)
