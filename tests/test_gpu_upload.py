"""swegl_scene_upload checks a whole description before it makes anything of
the sizes in it: one that names far more vertices than it has arrays for is
refused with SWEGL_EINVAL, and without memory for them."""
import ctypes as C
import resource

import pytest

from swegl_amd import _abi as A
from swegl_amd import host
from swegl_amd.device import Context, lib
from swegl_amd.host import SceneDescHolder

from test_oracle_scene import A_, B_, C_, flat_scene

pytestmark = pytest.mark.gpu
MANY = 400_000_000   # vertices: 12.8 GB of coordinates


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


def null_arrays(d):
    d.primitives[1].positions = A.FP()


def mode(d):
    d.primitives[1].mode = 7


def material(d):
    d.primitives[1].material_id = 5


def texture(d):
    d.materials[0].texture_idx = 3


def index(d):
    d.primitives[1].indices[2] = MANY


def range_of_primitives(d):
    d.nodes[1].n_primitives = 3


def empty_texture(d):
    d.textures[0].width = 0


@pytest.mark.parametrize("fault", [null_arrays, mode, material, texture, index, range_of_primitives, empty_texture])
def test_faulty_description_of_many_vertices(ctx, fault):
    s = flat_scene([[A_, B_, C_]])
    p = flat_scene([[A_, B_, C_]]).nodes[0].primitives[0]
    s.nodes.append(host.node_t([p]))
    h = SceneDescHolder(s)
    d = h.desc
    if fault is not empty_texture:   # the description is whole up to there
        d.primitives[1].n_vertices = MANY
    fault(d)
    before = resource.getrusage(resource.RUSAGE_SELF).ru_maxrss
    out = C.c_void_p()
    assert lib().swegl_scene_upload(ctx.h, C.byref(d), C.byref(out)) == A.EINVAL
    grown = (resource.getrusage(resource.RUSAGE_SELF).ru_maxrss - before) / 1e6   # GB
    assert grown < 1.0, f"{grown:.1f} GB for a refused description"
