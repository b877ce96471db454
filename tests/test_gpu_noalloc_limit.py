"""swegl_render_noalloc takes a render that fills its fixed array to the last
KB: the array's pieces, 256-byte aligned, are as large as the sizes below."""
import numpy as np
import pytest

import oracle
from swegl_amd.device import Context

from _helpers import compare, gpu_render
from test_oracle_scene import flat_scene, view

pytestmark = pytest.mark.gpu
ARRAY = 64 << 20
TRIANGLES, SIDE, TILE, BIN_LIMIT = 872_000, 64, 16, 16


def array_bytes(vertices):
    tiles = (SIDE // TILE) ** 2
    counters = 1024 + 8 * 64 + 64 + 33 * 32 + 2   # statistics, queues, totals, tickets, two words of the job
    used = 0
    for piece in (16 * vertices, vertices, 8 * TRIANGLES, 4 * TRIANGLES, 512, 128 * tiles + 8, 8 * tiles + 8,
                  4 * BIN_LIMIT * TRIANGLES, 4 * counters):
        used = (used + 255) // 256 * 256 + piece
    return used


def test_array_filled_to_the_last_kb():
    vertices = next(v for v in range(3, 1 << 20) if array_bytes(v) > ARRAY) - 1
    assert ARRAY - array_bytes(vertices) < 1024
    s = flat_scene([[[-0.5, -0.5, 0], [0.5, -0.5, 0], [0.0, 0.5, 0]]] + [[[0, 0, 9.0]] * 3])
    p = s.nodes[0].primitives[0]
    # one triangle in view, the others behind the camera; vertices of no
    # triangle fill the array up
    p.indices = np.concatenate([[0, 1, 2], np.full(3 * (TRIANGLES - 1), 3)]).astype(np.uint32)
    for name in ("positions", "normals", "tex_coords"):
        a = getattr(p, name)
        setattr(p, name, np.concatenate([a, np.repeat(a[-1:], vertices - len(a), 0)]))
    vp = view(SIDE, SIDE)
    ctx = Context(0)
    try:
        ctx.set_tile_auto(False)
        ctx.set_tile(TILE, TILE)
        ctx.set_bin_limit(BIN_LIMIT)
        got = gpu_render(ctx, s, [vp], with_tid=False, entry="swegl_render_noalloc")
    finally:
        ctx.close()
    compare(got[0], oracle.render(s, [vp])[0], check_tid=False)
