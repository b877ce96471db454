"""Tiles of more entries than are rasterised whole (their rows are then split
into bands) that also hold triangles of which the projected vertices do not
tell the rows: near-clipped ones, whose vertex behind the camera projects to
the wrong side, beside ones of depths far apart and far outside coordinates.
Depth bits, winners and fragment counts equal the oracle's."""
import numpy as np
import pytest

import oracle
from swegl_amd.device import Context

from _helpers import compare, gpu_render
from test_oracle_scene import flat_scene, view

pytestmark = pytest.mark.gpu
SIDE = 256   # the viewport; the crowd lies in rows 32-63, columns 128-159

# World points with the camera at z = 3, found by projecting random ones: every
# vertex projects below row 66, the triangle covers rows from 0 on and at most
# 14 tiles of 32x32.
NEAR = [[[0.382, 0.586, 4.751], [-0.185, 0.242, 4.922], [0.23, 0.488, 1.185]],
        [[-0.264, 0.086, 4.118], [0.559, 0.345, 3.263], [0.03, 0.217, 1.942]],
        [[-0.367, 0.068, 3.924], [0.116, -0.497, 4.676], [0.115, 0.491, 1.349]],
        [[-0.019, 0.51, 4.892], [-0.193, -0.445, 4.711], [0.106, 0.413, 1.107]]]


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


def crowd(rng, n):
    c = rng.uniform(-0.2, 0.2, (n, 1, 3)) * [1, 1, 0.5] + [0.329, 1.667, 0.0]
    return c + rng.uniform(-0.05, 0.05, (n, 3, 3))


def others(rng, kind, n):
    if kind == "near":
        return np.array(NEAR)[np.arange(n) % len(NEAR)] + rng.uniform(-0.002, 0.002, (n, 3, 3))
    t = crowd(rng, n) + rng.uniform(-0.1, 0.1, (n, 3, 3))
    if kind == "deep":
        t[:, 1] *= 14.0
        t[:, 1, 2] = -30.0
        t[:, 2] *= 0.3
        t[:, 2, 2] = 2.2
    else:
        assert kind == "wide"
        t[:, 2, 0] += rng.choice([-1.0, 1.0], n) * 10.0 ** rng.uniform(1, 6, n)
    return t


def vertex_rows(vp, tris):
    m = vp.m_camera.m_projectionmatrix.astype(np.float64) @ vp.m_camera.m_viewmatrix.astype(np.float64)
    q = np.concatenate([tris, np.ones(tris.shape[:2] + (1,))], -1) @ m.T
    return SIDE / 2 - SIDE / 2 * q[..., 1] / np.abs(q[..., 2])


@pytest.mark.parametrize("tile", [(32, 32), (64, 32), (64, 64)])
@pytest.mark.parametrize("n", [4, 300, 600])   # one list of 256 or 512 triangles holds them, or neither does
@pytest.mark.parametrize("kind", ["near", "deep", "wide"])
def test_bands_keep_triangles_that_are_not_plain(ctx, kind, n, tile):
    rng = np.random.default_rng(n + len(kind))
    odd = others(rng, kind, n)
    vp = view(SIDE, SIDE)
    if kind == "near":
        assert vertex_rows(vp, odd).min() > 64
        alone = oracle.render(flat_scene(odd.tolist(), double_sided=True), [vp])[0]
        assert (alone.tid[32:64, 128:160] != 0xFFFFFFFF).sum() > 300
    s = flat_scene(rng.permutation(np.concatenate([crowd(rng, 4500), odd])).tolist(), double_sided=True)
    want = oracle.render(s, [vp])[0]
    ctx.set_tile_auto(False)
    ctx.set_tile(*tile)
    try:
        got = gpu_render(ctx, s, [vp])[0]
    finally:
        ctx.set_tile_auto(True)
        ctx.set_tile(32, 32)
    compare(got, want)
    assert got.stats["fragments"] == want.stats["fragments"]
