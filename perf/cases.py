"""The renderer's work as its users call it, as cases that can be timed.

A case names an entry point (`call`), a synthetic scene of noor_amd.scenes with
its size, and the image or batch to compute:

  frame     Renderer.render: one call of the drop-in megakernel, the call a
            viewer makes for every displayed frame
  film      Renderer.render_wavefront: an offline film of `spp` samples
  batch     Renderer.render_batch: views of uneven size and sample count
  trace     Renderer.trace: hit queries on host arrays (picking, visibility)
  gradient  noor_amd.autograd.render, forward and backward
  build     SceneBuilder.build(device=...): trees of a new mesh on the GPU

The geometry belongs to the case; the seed draws what changes from call to
call: the camera, the rays, the parameters, or the mesh that is built.
"""
import ctypes as C
import functools
import math

import numpy as np
import torch

from noor_amd import abi, autograd, scenes
from noor_amd._lib import check, lib
from noor_amd.renderer import Renderer, rays_from_numpy
from noor_amd.scene import Mesh, SceneBuilder, make_camera, make_options, material

RNGS = {"pcg32": abi.RNG_PCG32, "tea_lcg": abi.RNG_TEA_LCG}
TRIS = {"watertight": abi.TRI_WATERTIGHT, "wald": abi.TRI_WALD}


def listed():
    return [
        # a thumbnail or material preview: a few thousand paths, so what counts is the call itself
        {"name": "frame_cornell_64", "call": "frame", "scene": "cornell", "detail": 4, "w": 64, "h": 64, "spp": 1,
         "bounces": 5},
        # the viewer on a small scene while the camera moves: new camera, a few samples per displayed frame
        {"name": "frame_cornell_512", "call": "frame", "scene": "cornell", "detail": 6, "w": 512, "h": 512, "spp": 4,
         "bounces": 5},
        # the viewer on the large scene (5M triangles, 1,000 instanced spheres, HDR environment) at full HD
        {"name": "frame_terrain_1080p", "call": "frame", "scene": "terrain", "detail": 1582, "w": 1920, "h": 1080,
         "spp": 1, "bounces": 8},
        # the small offline film: area light, diffuse box, 82k triangles
        {"name": "film_cornell_512", "call": "film", "scene": "cornell", "detail": 6, "w": 512, "h": 512, "spp": 16,
         "bounces": 5},
        # the headline film of the benchmark
        {"name": "film_terrain_1080p", "call": "film", "scene": "terrain", "detail": 1582, "w": 1920, "h": 1080,
         "spp": 32, "bounces": 8},
        # the benchmark's 1M-triangle scene of metal, glass and diffuse meshes under the physical sky
        {"name": "film_procedural_1080p", "call": "film", "scene": "procedural", "detail": 1000000, "w": 1920,
         "h": 1080, "spp": 64, "bounces": 8},
        # image textures, bump and alpha maps
        {"name": "film_textured_1080p", "call": "film", "scene": "textured", "detail": 512, "w": 1920, "h": 1080,
         "spp": 8, "bounces": 6},
        # every light type with multiple importance sampling, in the reference's own RNG and triangle test, odd size
        {"name": "film_lights_odd", "call": "film", "scene": "lights", "detail": 5, "w": 515, "h": 389, "spp": 16,
         "bounces": 6, "mis": True, "rng": "tea_lcg", "tri": "wald"},
        # a batch of uneven views (thumbnails to full HD, 1 to 64 samples) of one scene
        {"name": "batch_procedural_16", "call": "batch", "scene": "procedural", "detail": 1000000, "views": 16,
         "layout": 7, "bounces": 8},
        # visibility and picking queries from host code: an odd number of incoherent rays
        {"name": "trace_open_100k", "call": "trace", "scene": "open", "detail": 6, "rays": 100003, "any_hit": False,
         "bounces": 4},
        # one step of an optimiser over 64 materials and the environment: image, then its gradients
        {"name": "gradient_open_512", "call": "gradient", "scene": "open", "detail": 6, "w": 512, "h": 512,
         "bounces": 4},
        # a new mesh of half a million triangles becomes renderable
        {"name": "build_heightfield_513", "call": "build", "scene": "heightfield", "detail": 513},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _detail(rng, scene):
    if scene in ("cornell", "open", "lights"):
        return rng.randint(3, 6)
    if scene == "terrain":
        return _log(rng, 100, 700)
    if scene == "procedural":
        return _log(rng, 100000, 1000000)
    return 2 ** rng.randint(5, 9)  # texture sides of the textured scene


# samples of a drawn image or batch, at most: about the time of the largest listed case
MOST_SAMPLES = {"cornell": 30e6, "lights": 30e6, "textured": 30e6, "terrain": 60e6, "procedural": 130e6}


def draw(rng):
    while True:
        case = _draw(rng)
        if case["call"] == "batch":
            samples = sum(w * h * s for w, h, s in _batch_layout(case))
        else:
            samples = case.get("w", 0) * case.get("h", 0) * case.get("spp", 0)
        if samples <= MOST_SAMPLES.get(case["scene"], 1e9):
            return case


def _draw(rng):
    call = rng.choice(["frame", "frame", "film", "film", "film", "batch", "trace", "gradient", "build"])
    if call == "build":
        return {"call": call, "scene": "heightfield", "detail": _log(rng, 95, 600)}
    if call == "trace":
        scene = rng.choice(["open", "procedural", "terrain"])
        return {"call": call, "scene": scene, "detail": _detail(rng, scene), "rays": _log(rng, 100, 500000),
                "any_hit": rng.random() < 0.5, "bounces": 4}
    if call == "gradient":
        return {"call": call, "scene": "open", "detail": _detail(rng, "open"), "w": _log(rng, 48, 600),
                "h": _log(rng, 48, 600), "bounces": rng.randint(2, 5)}
    if call == "batch":
        scene = rng.choice(["procedural", "terrain"])
        return {"call": call, "scene": scene, "detail": _detail(rng, scene), "views": rng.randint(2, 12),
                "layout": rng.randint(0, 1 << 20), "bounces": rng.randint(3, 8)}
    scene = rng.choice(["cornell", "procedural", "terrain", "textured", "lights"])
    case = {"call": call, "scene": scene, "detail": _detail(rng, scene), "w": _log(rng, 33, 1920),
            "h": _log(rng, 31, 1080), "spp": _log(rng, 1, 8 if call == "frame" else 48), "bounces": rng.randint(2, 8)}
    if rng.random() < 0.25:
        case["rng"] = "tea_lcg"
    if rng.random() < 0.25:
        case["tri"] = "wald"
    if scene in ("lights", "textured") and rng.random() < 0.5:
        case["mis"] = True
    return case


# ----------------------------------------------------------------------------------------------
# scenes: the built payload of each geometry is kept, as a program keeps the scene it has loaded

@functools.lru_cache(maxsize=6)
def _workload(scene, detail, bounces, mis):
    if scene == "cornell":
        return scenes.cornell(subdiv=detail, bounces=bounces)
    if scene == "terrain":
        return scenes.terrain(grid=detail, bounces=bounces, build_device=0)
    if scene == "procedural":
        return scenes.procedural(target_tris=detail, bounces=bounces, build_device=0)
    if scene == "textured":
        return scenes.textured(tex=detail, bounces=bounces, mis=mis)
    if scene == "lights":
        return scenes.lights(subdiv=detail, bounces=bounces, mis=mis)
    return scenes.adjoint_scene(subdiv=detail, bounces=bounces)


# eye, look-at point and field of view (degrees) of each scene
VIEWS = {
    "cornell": ((0.0, 0.0, 0.95), (0.0, -0.1, -1.0), 60.0),
    "open": ((0.0, 0.0, 0.95), (0.0, -0.1, -1.0), 60.0),
    "lights": ((0.0, 0.0, 0.95), (0.0, -0.1, -1.0), 60.0),
    "textured": ((0.0, 0.0, 0.95), (0.0, -0.15, -1.0), 60.0),
    "terrain": ((0.0, 90.0, 480.0), (0.0, 0.0, 0.0), 50.0),
    "procedural": ((50.0, 75.0, 210.0), (50.0, 45.0, 50.0), 45.0),
}


def _camera(scene, w, h, g):
    """The scene's camera, turned by up to three degrees about the point it looks at."""
    eye, look, fov = VIEWS[scene]
    a = g.uniform(-0.05, 0.05)
    dx, dz = eye[0] - look[0], eye[2] - look[2]
    eye = (look[0] + dx * math.cos(a) + dz * math.sin(a), eye[1], look[2] - dx * math.sin(a) + dz * math.cos(a))
    return make_camera(eye, look, (0, 1, 0), math.radians(fov), w, h)


SIZES = ((256, 256), (512, 512), (1280, 720), (1920, 1080))
SPPS = (1, 4, 16, 64)


def _batch_layout(case):
    """(width, height, spp) of each view of a batch."""
    g = np.random.default_rng(case["layout"])
    return [SIZES[int(g.integers(4))] + (SPPS[int(g.integers(4))],) for _ in range(case["views"])]


def _batch_views(case, g):
    eye, look, _ = VIEWS[case["scene"]]
    dist = math.dist(eye, look)
    views = []
    for w, h, spp in _batch_layout(case):
        d = g.normal(size=3)
        d[1] = abs(d[1]) + 0.3
        d /= np.linalg.norm(d)
        cam = make_camera(tuple(np.asarray(look) + d * dist * g.uniform(0.7, 1.2)), look, (0, 1, 0),
                          math.radians(g.uniform(35.0, 60.0)), w, h)
        views.append((cam, 1, spp, int(g.integers(1 << 20))))
    return views


class _DeviceFilm:
    """A film in device memory for torch.as_tensor: what a viewer displays or a denoiser reads."""

    def __init__(self, ptr, w, h):
        self.__cuda_array_interface__ = {"shape": (h, w, 4), "typestr": "<f4", "data": (ptr, False), "version": 2}


def _film(renderer, ptr, w, h):
    film = torch.as_tensor(_DeviceFilm(ptr, w, h), device="cuda")
    film.renderer = renderer  # the owner of the memory lives as long as the tensor
    return film


class _PayloadArray(np.ndarray):
    """A view of a payload's memory that keeps the payload."""

    payload = None


def _payload_arrays(payload):
    out = {}
    for k, a in payload.arrays().items():
        out[k] = a.view(_PayloadArray)
        out[k].payload = payload
    return out


def _batch_film_ptr(r, i):
    p = C.c_void_p()
    check(lib().noor_batch_film_device_ptr(r._h, i, C.byref(p)), r._h)
    return p.value


def _rays(case, g):
    """Ray origins around the scene's centre and uniform directions."""
    eye, look, _ = VIEWS[case["scene"]]
    n = case["rays"]
    o = np.asarray(look, np.float64) + g.uniform(-0.5, 0.5, (n, 3)) * abs(eye[2] - look[2])
    if case["scene"] == "open":
        # above the block, whose base lies in the floor: two surfaces at one distance have no one answer
        o = g.uniform((-0.9, -0.15, -0.9), (0.9, 0.9, 0.9), (n, 3))
    if case["scene"] == "terrain":
        o[:, 1] = g.uniform(25.0, 60.0, n)
    d = g.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return o.astype(np.float32), d.astype(np.float32)


@functools.lru_cache(maxsize=4)
def _heightfield(n):
    return scenes.grid_heightfield(n, 100.0, lambda x, z: 8.0 * scenes.fbm2(x, z, 6, 5, 0.04))


def prepare(case, seed):
    g = np.random.default_rng([seed, 17])
    call, scene = case["call"], case["scene"]
    if call == "build":
        sb = SceneBuilder()
        sb.add_material(material(abi.MAT_DIFFUSE))
        # the mesh with its triangle list begun elsewhere, as another exporter would write it
        pos, tri, uv = _heightfield(case["detail"])
        sb.add_mesh(Mesh(pos, np.roll(tri, int(g.integers(1, len(tri))), axis=0), uvs=uv, material=0))
        return {"call": call, "builder": sb}
    wl = _workload(scene, case["detail"], case["bounces"], case.get("mis", False))
    opt = make_options(rng=RNGS[case.get("rng", "pcg32")], tri_test=TRIS[case.get("tri", "watertight")],
                       compat=wl.options.compat)
    w, h = case.get("w", 64), case.get("h", 64)
    cam = _camera(scene, w, h, g)
    r = Renderer(wl.payload, cam, wl.spec, opt, wl.hosek)
    state = {"call": call, "renderer": r, "camera": cam, "w": w, "h": h, "spp": case.get("spp", 1)}
    if call == "batch":
        state["views"] = _batch_views(case, g)
    elif call == "trace":
        state["rays"] = rays_from_numpy(*_rays(case, g))
        state["any_hit"] = case["any_hit"]
    elif call == "gradient":
        m = wl.info["n_materials"]
        dev = lambda a: torch.tensor(np.asarray(a, np.float32), device="cuda")  # noqa: E731
        state["albedo"] = dev(g.uniform(0.3, 0.7, (m, 3)))
        state["roughness"] = dev(g.uniform(0.2, 0.5, m))
        state["env"] = dev(wl.info["env"][..., :3] * g.uniform(0.8, 1.2, (1, 1, 3)))
        state["target"] = dev(g.uniform(0.0, 1.0, (h, w, 3)))
    return state


def run(state):
    call = state["call"]
    if call == "build":
        return _payload_arrays(state["builder"].build(device=0))
    r = state["renderer"]
    if call == "frame":
        r.update_camera(state["camera"])
        r.render(state["spp"])
        return _film(r, r.film_device_ptr(), state["w"], state["h"])
    if call == "film":
        r.render_wavefront(state["spp"], frame=1)
        return _film(r, r.film_device_ptr(), state["w"], state["h"])
    if call == "batch":
        r.render_batch(state["views"])
        return [_film(r, _batch_film_ptr(r, i), v[0].w, v[0].h) for i, v in enumerate(state["views"])]
    if call == "trace":
        hits = np.frombuffer(r.trace(state["rays"], any_hit=state["any_hit"]), np.uint32).reshape(-1, 8)
        return {"tuv": hits[:, :3].view(np.float32), "ids": hits[:, 3:7]}
    leaves = [state[k].clone().requires_grad_(True) for k in ("albedo", "roughness", "env")]
    image = autograd.render(r, 1, *leaves)
    loss = ((image - state["target"]) ** 2).sum()
    loss.backward()
    return [image.detach()] + [t.grad for t in leaves]


# ----------------------------------------------------------------------------------------------
# what a pass cannot do without

# Per sample: extension and shadow rays; per ray: four-box node visits and triangle tests, as the
# library's counters report them at the listed sizes.
EVENTS = {
    "cornell": (4.08, 3.26, 5.9, 4.2), "open": (2.5, 2.0, 3.8, 2.1), "lights": (3.04, 1.91, 5.8, 3.8),
    "textured": (3.03, 0.85, 4.2, 3.5), "terrain": (1.73, 0.62, 16.9, 2.1), "procedural": (1.15, 0.06, 8.0, 1.0),
}
NODE_FLOPS, TRI_FLOPS, SHADE_FLOPS = 100, 60, 200  # four boxes; one watertight test; one bounce's sampling


def work(case):
    if case["call"] == "build":
        n = case["detail"]
        tris, verts = 2 * (n - 1) ** 2, n * n
        # vertices with uv and indices in; per triangle attributes, three Wald records, its id and about one
        # 32-byte node out, per vertex position, normal and uv; a bin update per level of the tree
        return {"bytes": verts * 20 + tris * 12 + tris * (64 + 4 + 32) + verts * 40,
                "flops": tris * 30 * math.log2(max(tris, 2))}
    ext, shd, nodes, tests = EVENTS[case["scene"]]
    per_ray = nodes * NODE_FLOPS + tests * TRI_FLOPS
    if case["call"] == "trace":
        return {"bytes": 64 * case["rays"], "flops": case["rays"] * per_ray}
    if case["call"] == "batch":
        layout = _batch_layout(case)
        px, samples = sum(w * h for w, h, _ in layout), sum(w * h * s for w, h, s in layout)
    else:
        px = case["w"] * case["h"]
        samples = px * case.get("spp", 1)
    share = min(1.0, case["bounces"] / 5.0)  # short paths cast fewer rays
    rays = 1.0 + max(ext - 1.0, 0.0) * share + shd * share
    flops = samples * (rays * per_ray + (rays - shd * share) * SHADE_FLOPS)
    if case["call"] == "gradient":  # the replay traces the same paths; image, its gradient, the parameters and theirs
        return {"bytes": px * 16 * 3 + 2 * 4 * (512 * 256 * 3 + 64 * 4), "flops": 2 * flops}
    return {"bytes": px * 16, "flops": flops}


def exact(case, seed):
    """Closest hits in binary64 by testing every triangle.  Films and gradients have no such value: which light, lobe
    or box a path of theirs takes is decided in binary32, and in binary64 some paths part from it; a built payload is
    whole numbers; the larger scenes' queries would take too long."""
    if case["call"] != "trace" or case["scene"] != "open" or case["any_hit"]:
        return None
    wl = _workload(case["scene"], case["detail"], case["bounces"], False)
    a = wl.payload.arrays()
    if case["rays"] * len(a["attr"]) > 2e10:
        return None
    t64 = lambda x: torch.tensor(np.ascontiguousarray(x), device="cuda", dtype=torch.float64)  # noqa: E731
    g = np.random.default_rng([seed, 17])
    _camera(case["scene"], 64, 64, g)
    o, d = (t64(x) for x in _rays(case, g))
    v = t64(a["vertices"][:, :3])
    idx = torch.tensor(a["attr"][:, :3].astype(np.int64), device="cuda")
    p0 = v[idx[:, 0]]
    e1, e2 = v[idx[:, 1]] - p0, v[idx[:, 2]] - p0
    n, pe1, pe2 = torch.linalg.cross(e1, e2), torch.linalg.cross(p0, e1), torch.linalg.cross(p0, e2)
    out = torch.zeros((len(o), 3), dtype=torch.float64, device="cuda")
    for i in range(0, len(o), 512):
        # Moeller-Trumbore over all triangles, with the triple products written as dot products of per-triangle vectors
        oo, dd = o[i:i + 512], d[i:i + 512]
        m = torch.linalg.cross(oo, dd)  # moment of the ray
        det = -(dd @ n.T)
        u = (m @ e2.T + dd @ pe2.T) / det
        w = -(m @ e1.T + dd @ pe1.T) / det
        t = (oo @ n.T - (p0 * n).sum(1)) / det
        t = torch.where((u >= 0) & (w >= 0) & (u + w <= 1) & (t >= 0), t, torch.inf)
        best, k = t.min(dim=1)
        hit = torch.isfinite(best)
        at = lambda x: x.gather(1, k[:, None])[:, 0]  # noqa: E731
        res = torch.stack([best, at(u), at(w)], 1)
        out[i:i + 512] = torch.where(hit[:, None], res, torch.zeros_like(res))
    return {"tuv": out, "ids": None}
