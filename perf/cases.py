"""The renderer's workloads as measurable cases.

A case is a dict of plain values; `prepare` makes what a program holds before
it renders (a context, resident scenes, device surfaces, viewport
descriptions), `run` is one pass through the library's entry points, `work`
what that pass cannot do without, and `exact` the depth planes in 64 bits by
plain torch.  Scene kinds, sizes and options are those of the benchmark, the
autotuner and the tests: the cube, the reference demo's scene, height fields
of 10^3 to 10^6 triangles, stacked clusters in several viewports, mixed
batches and served streams.

Frames stay on the device, as in the benchmark's frame rates: an output is a
tensor over the surface that the render wrote.  Only the drop-in call reads
its frame back, because it leaves it in the caller's host surface.
"""
import ctypes as C
import math
import random

import numpy as np
import torch

from swegl_amd import _abi as A
from swegl_amd import autotune, host, scenes
from swegl_amd.device import Context, DeviceScene, Server, Target, check, lib

NEAR = 0.001
MAX_Z = float(np.uint32(0x7F7F7F7F).view(np.float32))   # the cleared depth plane

LIGHTS = {"phong": host.pixel_shader_lights_phong, "flat": host.pixel_shader_lights_flat}
TEXTURES = {"bilinear": host.pixel_shader_texture_bilinear, "nearest": host.pixel_shader_texture}
ALONE = {"material": host.pixel_shader_t, "texture_nearest": host.pixel_shader_texture,
         "texture_bilinear": host.pixel_shader_texture_bilinear,
         "lights_flat": host.pixel_shader_lights_flat, "lights_phong": host.pixel_shader_lights_phong}
SHADERS = [l + "_" + t for l in LIGHTS for t in TEXTURES] + list(ALONE)


# ------------------------------------------------------------------ cases
def _field(name, n, width, height, tex, lights, shader="phong_bilinear", post="none", radius=0, entry="render"):
    return {"name": name, "kind": "field", "n": n, "width": width, "height": height, "tex_w": tex[0], "tex_h": tex[1],
            "lights": lights, "shader": shader, "post": post, "radius": radius, "entry": entry}


def listed():
    return [
        # one small object in a window, frame after frame: 12 triangles, so
        # the calls, launches and the shading of large triangles count
        {"name": "cube", "kind": "cube", "width": 640, "height": 480, "entry": "render"},
        # the reference's own call on a small window: scene described, posed,
        # rendered and read back into the caller's surface on every call
        {"name": "cube_dropin", "kind": "cube", "width": 320, "height": 240, "entry": "dropin"},
        # a small odd-sized preview replayed as a graph, ragged texture
        _field("field_small_graph", 64, 333, 251, (300, 170), 1, entry="graph"),
        # the reference demo's scene: strips, mid-size overlapping triangles
        {"name": "demo", "kind": "demo", "width": 800, "height": 600, "precision": 100, "layers": 0},
        # the same as the demo draws it, with its three transparency layers
        {"name": "demo_layers", "kind": "demo", "width": 800, "height": 600, "precision": 100, "layers": 3},
        # an animated object: a new pose before every frame, no post pass
        _field("field_posed", 317, 1280, 720, (1024, 1024), 2, entry="posed"),
        # the flat, unfiltered look with the reference's box blur, odd sizes
        _field("field_flat_box", 253, 1231, 717, (512, 512), 3, shader="flat_nearest", post="box", radius=5),
        # the benchmark's frame: a million small triangles at 1080p
        _field("field_1080p", 708, 1920, 1080, (2048, 2048), 4, post="tap9", radius=8),
        # the largest single view: 4K, wide blur
        _field("field_4k", 708, 3840, 2160, (2048, 2048), 4, post="tap9", radius=16),
        # half a million stacked triangles seen by four cameras in one call
        {"name": "heavy_views", "kind": "heavy", "clusters": 500, "views": 4, "width": 1920, "height": 1080,
         "tex": 4096, "lights": 8, "radius": 8},
        # many independent scenes in one call
        {"name": "batch", "kind": "batch", "count": 32, "mix": 1, "tmin": 1000, "tmax": 200000},
        # a burst of requests to the server: mixed scenes and a few large frames
        {"name": "served", "kind": "served", "count": 30, "mix": 2, "tmin": 1000, "tmax": 200000, "large": 2},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["field", "graph", "posed", "cube", "demo", "heavy", "batch", "served"],
                       [8, 3, 2, 2, 3, 2, 2, 2])[0]
    if kind in ("field", "graph", "posed"):
        w = _log(rng, 64, 2560)
        h = max(48, min(2160, int(w * rng.uniform(0.4, 1.1))))
        post = rng.choice(["none", "none", "box", "tap9"])
        # captured graphs hold depth of field with the Phong and bilinear
        # shader only; half of all frames use that shader anyway
        shader = "phong_bilinear" if kind == "graph" or rng.random() < 0.5 else rng.choice(SHADERS)
        return _without_name(_field("", _log(rng, 24, 708), w, h, (_log(rng, 16, 2048), _log(rng, 16, 2048)),
                                    rng.randint(0, 8), shader, post,
                                    rng.randint(1, 16 if post == "tap9" else 8) if post != "none" else 0,
                                    {"field": "render"}.get(kind, kind)))
    if kind == "cube":
        w = _log(rng, 96, 1920)
        return {"kind": "cube", "width": w, "height": max(64, int(w * rng.uniform(0.5, 1.0))),
                "entry": rng.choice(["render", "render", "graph", "dropin"]) if w <= 800 else "render"}
    if kind == "demo":
        w = _log(rng, 160, 1280)
        return {"kind": "demo", "width": w, "height": max(120, int(w * rng.uniform(0.5, 1.0))),
                "precision": _log(rng, 12, 120), "layers": rng.randint(0, 4)}
    if kind == "heavy":
        w = _log(rng, 320, 1920)
        return {"kind": "heavy", "clusters": _log(rng, 20, 500), "views": rng.randint(1, 4), "width": w,
                "height": max(180, int(w * rng.uniform(0.45, 0.6))), "tex": _log(rng, 256, 4096),
                "lights": rng.randint(1, 8), "radius": rng.choice([0, 3, 5, 8])}
    c = {"kind": kind, "count": rng.randint(4, 30), "mix": rng.randrange(1 << 20), "tmin": 1000,
         "tmax": _log(rng, 4000, 200000)}
    if kind == "served":
        c["large"] = rng.randint(0, min(2, c["count"] // 8))
    return c


def _without_name(c):
    del c["name"]
    return c


# ----------------------------------------------------------------- inputs
def _field_job(c, seed):
    scene, vps = scenes.heightfield_scene(seed, n=c["n"], width=c["width"], height=c["height"], tex=1,
                                          n_lights=c["lights"], dof=False)
    scene.images = [scenes.random_texture(np.random.default_rng(seed + 1), c["tex_w"], c["tex_h"])]
    vp = vps[0]
    if c["shader"] in ALONE:
        vp.m_pixel_shader = ALONE[c["shader"]]()
    else:
        light, texture = c["shader"].split("_")
        vp.m_pixel_shader = host.pixel_shader_light_and_texture(LIGHTS[light], TEXTURES[texture])
    if c["post"] != "none":
        vp.set_post_shader(host.post_shader_depth_box(5.0, 5.0, vp, max_radius=c["radius"], taps=c["post"]))
    if c["entry"] == "posed":
        a = random.Random(seed).uniform(-0.4, 0.4)
        scene.nodes[0].rotation = host.rotate_y(host.IDENTITY.copy(), a)
    return scene, vps


def _mixed(c):
    """The height fields of a batch or stream: triangle counts spread over
    their logarithm, the benchmark's sides, texture sizes and lights, the
    9-tap blur on half of them, and `large` frames of a million triangles."""
    r = random.Random(c["mix"])
    out = []
    for k in range(c["count"]):
        t = math.exp(r.uniform(math.log(c["tmin"]), math.log(c["tmax"])))
        side = r.choice([256, 384, 512, 768, 1024])
        tex = r.choice([512, 1024])
        dof = k % 2 == 0
        out.append(_field("", int(round(math.sqrt(t / 2.0))) + 1, side, side, (tex, tex), r.randint(0, 4),
                          post="tap9" if dof else "none", radius=8 if dof else 0))
    for k in range(c.get("large", 0)):
        out[(k + 1) * len(out) // (c["large"] + 1)] = _field("", 708, 1920, 1080, (2048, 2048), 4, post="tap9",
                                                              radius=8)
    return out


def _jobs(c, seed):
    """The case's (scene, viewports) pairs, from the seed alone."""
    if c["kind"] == "cube":
        return [scenes.cube_scene(seed, c["width"], c["height"])]
    if c["kind"] == "demo":
        s = scenes.demo_scene(seed, c["precision"], c["precision"])
        s.nodes[0].rotation = host.rotate_z(host.IDENTITY.copy(), random.Random(seed).uniform(0.2, 0.8))
        return [(s, [scenes.demo_viewport(c["width"], c["height"], c["layers"])])]
    if c["kind"] == "field":
        return [_field_job(c, seed)]
    if c["kind"] == "heavy":
        return [scenes.heavy_scene(seed, c["clusters"], c["views"], c["width"], c["height"], c["tex"], c["lights"],
                                   dof=c["radius"] > 0, dof_radius=c["radius"])]
    return [_field_job(f, seed + 7919 * k) for k, f in enumerate(_mixed(c))]


class _Device:
    """A target's memory for torch, which keeps the target alive with the
    tensor.  The library hands out no device address, so it is read from the
    head of the target's record: kind, width, height, address, bytes."""

    def __init__(self, target):
        self.target = target
        kind, w, h = (C.c_int32 * 3).from_address(target.h.value)
        p, n = (C.c_uint64 * 2).from_address(target.h.value + 16)
        if (kind, w, h, n) != (target.kind, target.width, target.height, max(256, 4 * w * h)):
            raise RuntimeError("swegl_target is laid out in another way than expected")
        self.__cuda_array_interface__ = {"shape": (h, w), "typestr": "<f4" if kind == A.TARGET_FLOAT else "<i4",
                                         "data": (p, False), "version": 2, "strides": None}


def _tensor(target):
    return torch.as_tensor(_Device(target), device="cuda")


_contexts = {}


def _context(c):
    """One context for single renders and one for batches and streams, each
    with its tuned settings, as the benchmark runs them."""
    key = "batch" if c["kind"] in ("batch", "served") else "heightfield"
    if key not in _contexts:
        ctx = Context(0)
        ctx.apply_tuning(autotune.load()[key])
        _contexts[key] = ctx
    return _contexts[key]


def prepare(case, seed):
    ctx, jobs = _context(case), _jobs(case, seed)
    st = {"case": case, "ctx": ctx, "jobs": jobs}
    if case.get("entry") == "dropin":
        return st
    st["scenes"], st["descs"], st["out"], st["holders"] = [], [], [], []
    arr = (A.Job * len(jobs))()
    for k, (scene, vps) in enumerate(jobs):
        holder = host.SceneDescHolder(scene)
        ds = DeviceScene(ctx, holder)
        d = (A.ViewportDesc * len(vps))()
        for i, vp in enumerate(vps):
            color = Target(ctx, A.TARGET_COLOR, vp.m_screen.w, vp.m_screen.h)
            depth = Target(ctx, A.TARGET_FLOAT, vp.m_w, vp.m_h)
            d[i] = vp.desc(color, depth)
            st["out"].append({"color": _tensor(color), "depth": _tensor(depth)})
        st["holders"].append(holder)
        st["scenes"].append(ds)
        st["descs"].append(d)
        arr[k] = A.Job(ds.h, d, len(vps))
    st["arr"] = arr
    if case["kind"] == "served":
        st["server"] = Server(ctx, 64 << 30, max_batch=64, lanes=3)
    return st


# -------------------------------------------------------------------- run
def run(state):
    case, ctx, L = state["case"], state["ctx"], lib()
    entry = case.get("entry", "render")
    if entry == "dropin":
        scene, vps = state["jobs"][0]
        host.render(scene, *vps, ctx=ctx)
        return [{"color": vp.m_screen.pixels.view(np.int32), "depth": vp.m_zbuffer.reshape(vp.m_h, vp.m_w)}
                for vp in vps]
    if case["kind"] == "batch":
        check(L.swegl_render_batch_graph(ctx.h, state["arr"], len(state["arr"]), None), "swegl_render_batch_graph")
    elif case["kind"] == "served":
        for job in state["arr"]:
            state["server"].submit(job)
        state["server"].drain()
        state["server"].poll()
    else:
        ds, d = state["scenes"][0], state["descs"][0]
        if entry == "posed":
            ds.update_pose(state["holders"][0])
        fn = L.swegl_render_graph if entry == "graph" else L.swegl_render
        check(fn(ctx.h, ds.h, d, len(d), None), "swegl_render")
    return state["out"]


# ------------------------------------------------------------------- work
def _shape(c):
    """(vertices, triangles, texture bytes, lights, pixels of each viewport)."""
    if c["kind"] == "cube":
        return 24, 12, 256 * 256 * 4, 0, [c["width"] * c["height"]]
    if c["kind"] == "demo":
        n = c["precision"] + 1
        return 4 * n * n + 81, 4 * n * c["precision"] + 39, 3 * 256 * 256 * 4, 2, [c["width"] * c["height"]]
    if c["kind"] == "heavy":
        return (c["clusters"] * 26 * 21, c["clusters"] * 1000, c["tex"] * c["tex"] * 4, c["lights"],
                [c["width"] * c["height"]] * c["views"])
    return c["n"] * c["n"], 2 * (c["n"] - 1) ** 2, c["tex_w"] * c["tex_h"] * 4, c["lights"], [c["width"] * c["height"]]


def work(case):
    """Bytes: a scene's vertices (32) and indices (12 a triangle) once, the
    texels at most once each and at most four a pixel, colour and depth
    written.  Operations: two transforms of each vertex and about 60 a
    triangle per viewport, about 150 a pixel and 50 for each light on it, if
    half of the pixels are covered."""
    nbytes = flops = 0
    for c in _mixed(case) if case["kind"] in ("batch", "served") else [case]:
        v, t, tex, lights, pixels = _shape(c)
        p = sum(pixels)
        nbytes += 32 * v + 12 * t + min(tex, 16 * p) + 8 * p
        flops += len(pixels) * (36 * v + 60 * t) + p // 2 * (150 + 50 * lights)
    return {"bytes": nbytes, "flops": flops}


# ------------------------------------------------------------------ exact
def _triangles(p):
    """A primitive's triangles in the reference's order and winding."""
    i = p.indices.astype(np.int64)
    if p.mode == A.TRIANGLES:
        return i[:len(i) // 3 * 3].reshape(-1, 3)
    if p.mode == A.TRIANGLE_FAN:
        return np.stack([np.full(len(i) - 2, i[0]), i[1:-1], i[2:]], -1)
    t = np.stack([i[:-2], i[1:-1], i[2:]], -1)
    t[1::2] = t[1::2][:, [0, 2, 1]]
    return t


def _world(scene, dev):
    """World positions, triangles and, for each triangle, whether its
    material is opaque, in 64 bits (root nodes only)."""
    pos, tri, opaque, base = [], [], [], 0
    for nd in scene.nodes:
        m = np.asarray(nd.rotation, np.float64)[:3, :3] * np.asarray(nd.scale, np.float64)
        for p in nd.primitives:
            t = _triangles(p)
            mat = scene.materials[p.material_id]
            pos.append(p.positions.astype(np.float64) @ m.T + np.asarray(nd.translation, np.float64))
            tri.append(t + base)
            opaque.append(np.full(len(t), mat.texture_idx >= 0 or mat.color >> 24 == 255))
            base += len(p.positions)
    to = lambda x: torch.from_numpy(np.concatenate(x)).to(dev)  # noqa: E731
    return to(pos), to(tri), to(opaque)


def _spread(counts):
    """For each item of runs of the given lengths: its run and its place in it."""
    run_of = torch.repeat_interleave(torch.arange(len(counts), device=counts.device), counts)
    first = torch.cumsum(counts, 0) - counts
    return run_of, torch.arange(len(run_of), device=counts.device) - first[run_of]


def _depth(pos, tri, opaque, vp):
    """The viewport's depth plane: triangles whose three vertices belong to
    triangles in view and facing the camera, rows ceil(y0) <= y < ceil(y2),
    columns ceil(left) <= x < ceil(right), 1 / z linear on the screen, the
    smallest z at each pixel.  None if a triangle crosses the near plane."""
    cam = vp.m_camera
    view, proj = (torch.from_numpy(np.asarray(m, np.float64)).to(pos) for m in (cam.m_viewmatrix, cam.m_projectionmatrix))
    f = (pos @ view[:3, :3].T + view[:3, 3]) @ proj[:3, :3].T + proj[:3, 3]
    z = f[:, 2]
    ndc = f[:, :2] / z.abs().clamp_min(1e-300)[:, None]
    a, b, c = (ndc[tri[:, k]] for k in range(3))
    az = z[tri]
    lo, hi = torch.minimum(torch.minimum(a, b), c), torch.maximum(torch.maximum(a, b), c)
    inside = ((hi >= -1) & (lo < 1) & (lo != hi)).all(1) & (az >= NEAR).any(1)
    e, g = b - a, c - a
    marks = torch.zeros(len(pos), dtype=torch.bool, device=pos.device)
    marks[tri[inside & (e[:, 0] * g[:, 1] - e[:, 1] * g[:, 0] > 0)].reshape(-1)] = True
    drawn = marks[tri].all(1)
    if bool(((az < NEAR).any(1) & drawn).any()):
        return None
    tri = tri[drawn & opaque] if vp.transparency_layer_count else tri[drawn]
    x = (ndc[:, 0] * (vp.m_w / 2.0) + vp.m_x + vp.m_w / 2.0)[tri]
    y = (ndc[:, 1] * (-vp.m_h / 2.0) + vp.m_y + vp.m_h / 2.0)[tri]
    iz = (1.0 / z)[tri]
    y, order = y.sort(1)
    x, iz = x.gather(1, order), iz.gather(1, order)
    out = torch.full((vp.m_h * vp.m_w,), MAX_Z, dtype=torch.float64, device=pos.device)
    for part in torch.arange(len(tri), device=pos.device).split(1 << 17):
        px, py, pi = x[part], y[part], iz[part]
        y0 = py[:, 0].ceil().clamp_min(vp.m_y)
        rows = (py[:, 2].ceil().clamp_max(vp.m_y + vp.m_h) - y0).clamp_min(0).long()
        t, r = _spread(rows)
        row = y0[t] + r
        px, py, pi = px[t], py[t], pi[t]
        low = row >= py[:, 1].ceil()   # the short side is v1-v2 there, v0-v1 above
        k0, k1 = low.long()[:, None], low.long()[:, None] + 1
        at = lambda v, k: v.gather(1, k)[:, 0]  # noqa: E731
        s = (row - py[:, 0]) / (py[:, 2] - py[:, 0])
        u = (row - at(py, k0)) / (at(py, k1) - at(py, k0))
        lx, li = px[:, 0] + s * (px[:, 2] - px[:, 0]), pi[:, 0] + s * (pi[:, 2] - pi[:, 0])
        sx, si = at(px, k0) + u * (at(px, k1) - at(px, k0)), at(pi, k0) + u * (at(pi, k1) - at(pi, k0))
        swap = lx > sx
        xl, xr = torch.where(swap, sx, lx), torch.where(swap, lx, sx)
        il, ir = torch.where(swap, si, li), torch.where(swap, li, si)
        x0 = xl.ceil().clamp_min(vp.m_x)
        cols = (xr.ceil().clamp_max(vp.m_x + vp.m_w) - x0).clamp_min(0).long()
        q, d = _spread(cols)
        col = x0[q] + d
        zz = 1.0 / (il[q] + (col - xl[q]) / (xr[q] - xl[q]) * (ir[q] - il[q]))
        ok = zz >= NEAR
        place = ((row[q] - vp.m_y) * vp.m_w + (col - vp.m_x)).long()
        out.scatter_reduce_(0, place[ok], zz[ok], "amin")
    return out.reshape(vp.m_h, vp.m_w)


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    out = []
    for scene, vps in _jobs(case, seed):
        pos, tri, opaque = _world(scene, dev)
        for vp in vps:
            out.append({"color": None, "depth": _depth(pos, tri, opaque, vp)})
    return out
