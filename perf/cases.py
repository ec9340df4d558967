"""Performance cases: the work a program has this package do, through keepsake_amd.api.

The package renders triangle scenes with the small_pt path tracer (plain, batched over many views, or
guided by an online-trained network), answers ray queries, and builds its BVH on the device. A program
opens one device, uploads its scenes once and then renders frame after frame, so `prepare` takes the
device and the scenes from this module (made on first use and kept) and makes what belongs to a frame: a
film, a camera moved by the seed, the sampler's seed, a guide with its weights, a mesh that has moved.

Case kinds:
  render    film clear, ks_small_pt_render, composite (what the small_pt task does per progress interval)
  batch     many views of one scene in one call, each view's film composited
  guided    a render with a trained, frozen guide (inference in BF16 or FP8)
  train     the first pass of a guided render: one sample per pixel, training records, Adam steps
  gradient  the guide's loss and gradient on given samples (forward and backward)
  build     a scene whose mesh has moved: upload, device BVH build, closest-hit and occlusion queries
"""

from __future__ import annotations

import math

import numpy as np
import torch

from keepsake_amd import api as ks

# ------------------------------------------------------------------------------------------------
# Cases
# ------------------------------------------------------------------------------------------------


def listed():
    return [
        # a thumbnail: one sample per pixel of the smallest scene, where launches and waits count
        dict(name="preview_64", kind="render", scene="cornell", width=64, height=64, spp=1, bounces=8),
        # the Cornell box at its usual test size (256 x 256, 16 spp, depth 8); the sums are downloaded,
        # as a program that adds the samples of several processes does
        dict(name="cornell_256", kind="render", scene="cornell", width=256, height=256, spp=16, bounces=8,
             output="sums"),
        # the benchmark's frame: 1.31 M triangles under an ambient sky, glossy and metal spheres
        dict(name="spheres_1080p", kind="render", scene="spheres", width=1920, height=1080, spp=64, bounces=12),
        # one progress interval of a progressive 720p render of the slit-lit room: long indirect paths
        dict(name="room_720p", kind="render", scene="room", width=1280, height=720, spp=8, bounces=16,
             mis="consistent", clamp_indirect=0.0),
        # textured fields, a normal map and alpha-tested leaves, an odd frame size
        dict(name="textured_509x383", kind="render", scene="foliage", width=509, height=383, spp=16, bounces=8),
        # an environment map over a device-built BVH, a cropped window of an odd frame, the gaussian
        # pixel filter and a backdrop where nothing is hit
        dict(name="skymap_crop", kind="render", scene="skymap", width=1001, height=563, spp=4, bounces=5,
             crop=True, filter="gaussian", background=False),
        # camera views of uneven size in one call (turntables, light probes)
        dict(name="batch_12", kind="batch", scene="cornell", views=12, layout=0, bounces=12),
        # rendering with a trained guide: BF16 inference at the camera rays' hits
        dict(name="guided_720p_bf16", kind="guided", scene="room", width=1280, height=720, spp=8, bounces=16,
             fp8=False, max_bounce=1, fraction=0.3),
        # the same with FP8 inference at every vertex, an odd frame size
        dict(name="guided_801x451_fp8", kind="guided", scene="room", width=801, height=451, spp=8, bounces=16,
             fp8=True, max_bounce=0, fraction=0.5),
        # a training pass of a guided 720p render: the samples of its paths, 8 Adam steps of 2^18
        dict(name="train_720p", kind="train", scene="room", width=1280, height=720, bounces=16, steps=8,
             log2_table=16),
        # the guide trained from a program's own samples: one batch at the default table size
        dict(name="gradient_2e18", kind="gradient", scene="room", samples=262144, log2_table=19),
        # an animated mesh: 1.31 M triangles uploaded and built on the device, 2^18 rays of each kind
        dict(name="build_1m", kind="build", scene="spheres", rays=262144),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["render"] * 5 + ["batch", "guided", "train", "gradient", "build"])
    if kind == "render":
        scene = rng.choice(["cornell", "spheres", "room", "foliage", "skymap"])
        w, h = _log_int(rng, 48, 1600), _log_int(rng, 48, 1000)
        spp = rng.choice([1, 2, 3, 4, 6, 8, 12, 16, 32])
        spp = max(1, min(spp, 12_000_000 // (w * h)))  # at most 12 M paths: below the 1080p frame's work
        c = dict(kind=kind, scene=scene, width=w, height=h, spp=spp, bounces=rng.randint(2, 16))
        if rng.random() < 0.3:
            c["mis"] = "consistent"
        if rng.random() < 0.3:
            c["filter"] = rng.choice(["gaussian", "blackman_harris"])
        if rng.random() < 0.3:
            c["crop"] = True
        if rng.random() < 0.3:
            c["background"] = False
        if rng.random() < 0.3:
            c["output"] = "sums"
        return c
    if kind == "batch":
        return dict(kind=kind, scene="cornell", views=rng.randint(2, 14), layout=rng.randint(1, 10**6),
                    bounces=rng.randint(4, 12))
    if kind == "guided":
        w, h = _log_int(rng, 64, 1280), _log_int(rng, 64, 720)
        return dict(kind=kind, scene="room", width=w, height=h, spp=rng.choice([1, 2, 4, 5, 8]),
                    bounces=rng.randint(4, 16), fp8=rng.random() < 0.5, max_bounce=rng.choice([0, 1, 2, 3]),
                    fraction=rng.choice([0.2, 0.3, 0.5]))
    if kind == "train":
        return dict(kind=kind, scene="room", width=_log_int(rng, 128, 1280), height=_log_int(rng, 96, 720),
                    bounces=rng.randint(4, 16), steps=rng.randint(1, 8), log2_table=rng.choice([14, 15, 16]))
    if kind == "gradient":
        return dict(kind=kind, scene="room", samples=_log_int(rng, 64, 262144), log2_table=rng.choice([14, 16, 19]))
    return dict(kind=kind, scene=rng.choice(["spheres", "spheres_small", "room"]), rays=_log_int(rng, 1024, 262144))


# ------------------------------------------------------------------------------------------------
# What a program keeps: the device and the uploaded scenes
# ------------------------------------------------------------------------------------------------
_kept: dict = {}


def _device():
    if "device" not in _kept:
        _kept["device"] = ks.Device(0)
    return _kept["device"]


def _host_scene(name):
    key = ("host", name)
    if key not in _kept:
        if name == "foliage":
            _kept[key] = _foliage()
        elif name == "skymap":
            _kept[key] = _under_sky_map(_host_scene("spheres"))
        else:
            _kept[key] = ks.procedural_scene(name, {"spheres": 1, "spheres_small": 1, "room": 3}.get(name, 0))
    return _kept[key]


def _scene(name):
    key = ("scene", name)
    if key not in _kept:
        _kept[key] = ks.Scene(_device(), _host_scene(name), bvh={"builder": 1} if name == "skymap" else None)
    return _kept[key]


def _under_sky_map(base):
    """The spheres under a 512 x 256 HDR sky with a small sun in place of the ambient light."""
    h, w = 256, 512
    th = (np.arange(h) + 0.5) / h * np.pi
    ph = (np.arange(w) + 0.5) / w * 2 * np.pi
    up = np.cos(th)[:, None]
    grad = 0.2 + 0.6 * np.clip(up, 0, 1)[..., None] * np.asarray([0.5, 0.7, 1.0])
    sky = np.broadcast_to(grad, (h, w, 3)).copy()
    d = (th[:, None] - 0.9) ** 2 + (ph[None, :] - 2.1) ** 2
    sky += 60.0 * np.exp(-d / 0.004)[..., None] * np.asarray([1.0, 0.9, 0.7])
    lights = np.zeros(1, ks.LIGHT_DTYPE)
    lights["type"] = ks.KS_LIGHT_SKY_MAP
    return ks.HostScene(base.vertices, base.indices, base.tri_geom, base.geom_material, base.materials, lights,
                        dict(base.camera), sky_map=dict(rgb=sky.astype(np.float32), y_up=True, strength=1.0))


def _foliage():
    """A unit room with a tiled sRGB floor, a normal-mapped wall, a glossy wall with a roughness texture
    and 3000 alpha-tested leaf quads under a ceiling light."""
    rng = np.random.default_rng(11)
    v, tc, idx, tg, gm = [], [], [], [], []

    def quad(p, uv, geom):
        b = len(v)
        v.extend(p)
        tc.extend(uv)
        idx.extend([[b, b + 1, b + 2], [b, b + 2, b + 3]])
        tg.extend([geom, geom])

    unit = [(0, 0), (1, 0), (1, 1), (0, 1)]
    quad([(0, 0, 0), (0, 0, 1), (1, 0, 1), (1, 0, 0)], [(0, 0), (0, 4), (4, 4), (4, 0)], 0)  # floor
    quad([(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0)], unit, 1)  # back
    quad([(1, 0, 0), (1, 0, 1), (1, 1, 1), (1, 1, 0)], unit, 2)  # right
    quad([(0, 0, 0), (0, 1, 0), (0, 1, 1), (0, 0, 1)], unit, 3)  # left
    quad([(0, 1, 0), (0, 1, 1), (1, 1, 1), (1, 1, 0)], unit, 3)  # ceiling
    quad([(0.35, 0.998, 0.35), (0.65, 0.998, 0.35), (0.65, 0.998, 0.65), (0.35, 0.998, 0.65)], unit, 4)  # light
    for _ in range(3000):
        c = rng.uniform([0.1, 0.03, 0.1], [0.9, 0.7, 0.9])
        a = rng.normal(size=3)
        a /= np.linalg.norm(a)
        b = np.cross(a, rng.normal(size=3))
        b /= np.linalg.norm(b)
        s = rng.uniform(0.01, 0.03)
        quad([tuple(c - s * a - s * b), tuple(c + s * a - s * b), tuple(c + s * a + s * b),
              tuple(c - s * a + s * b)], unit, 5)
    gm = [0, 1, 2, 3, 4, 5]
    mats = np.zeros(6, ks.MATERIAL_DTYPE)
    mats["basecolor"], mats["roughness"], mats["ior"], mats["specular_r0_mul"] = 0.7, 0.6, 1.5, 0.5
    mats[4]["basecolor"], mats[4]["has_emission"], mats[4]["emission"] = 0.0, 1, (12.0, 11.0, 9.0)
    y, x = np.mgrid[0:128, 0:128]
    check = np.where(((x // 16 + y // 16) % 2 == 0)[..., None], (230, 215, 200), (30, 40, 80)).astype(np.uint8)
    ny, nx = np.mgrid[0:96, 0:96] / 96.0 * 6 * np.pi
    bump = np.stack([0.3 * np.sin(nx), 0.3 * np.cos(ny), np.ones_like(nx)], -1)
    bump /= np.linalg.norm(bump, axis=-1, keepdims=True)
    rough = (0.05 + 0.6 * (np.mgrid[0:40, 0:30][1] / 29.0)).astype(np.float32)[..., None]
    leaf = np.where(((x - 64) / 30.0) ** 2 + ((y - 64) / 60.0) ** 2 < 1.0, 255, 0).astype(np.uint8)[..., None]
    textures = [dict(data=check, srgb=True, mipmaps=True),
                dict(data=np.round((bump * 0.5 + 0.5) * 65535).astype(np.uint16), srgb=False, mipmaps=False),
                dict(data=rough, srgb=False, mipmaps=True), dict(data=leaf, srgb=False, mipmaps=False)]
    f = ks.field_desc
    fields = {
        0: ks.material_fields(mats[0], basecolor=f(texture=0, sampler=ks.KS_SAMPLER_EWA)),
        1: ks.material_fields(mats[1], normal_map=f(texture=1, sampler=ks.KS_SAMPLER_LINEAR), normal_strength=0.8),
        2: ks.material_fields(mats[2], roughness=f(texture=2, sampler=ks.KS_SAMPLER_CUBIC)),
        5: ks.material_fields(mats[5], basecolor=f(value=(0.2, 0.6, 0.25)),
                              opacity=f(texture=3, sampler=ks.KS_SAMPLER_NEAREST, swizzle=(0,))),
    }
    return ks.HostScene(
        vertices=np.asarray(v, np.float32), indices=np.asarray(idx, np.uint32), tri_geom=np.asarray(tg, np.uint32),
        geom_material=np.asarray(gm, np.uint32), materials=mats, lights=np.zeros(0, ks.LIGHT_DTYPE),
        camera=dict(pos=(0.5, 0.5, 2.2), target=(0.5, 0.45, 0.4), up=(0.0, 1.0, 0.0), vfov=42.0, aspect=1.0),
        texcoords=np.asarray(tc, np.float32), textures=textures, material_fields=fields)


# ------------------------------------------------------------------------------------------------
# Inputs of a pass
# ------------------------------------------------------------------------------------------------
class _State(dict):
    """A frame's films and guide; their device memory goes with the state."""

    def __del__(self):
        for handle in self.get("owned", ()):
            handle.close()


def _camera(name, rng, aspect):
    """The scene's camera, moved a little by the seed."""
    cam = dict(_host_scene(name).camera)
    size = {"cornell": 0.1, "foliage": 0.1, "room": 0.3}.get(name, 1.0)
    cam["pos"] = tuple(float(p + size * rng.uniform(-1, 1)) for p in cam["pos"])
    cam["aspect"] = aspect
    return cam


_FILTERS = {"box": ks.KS_FILTER_BOX, "gaussian": ks.KS_FILTER_GAUSSIAN,
            "blackman_harris": ks.KS_FILTER_BLACKMAN_HARRIS}
_BACKDROP = (0.1, 0.2, 0.3)


def _params(case, rng, spp):
    w, h = case["width"], case["height"]
    crop = dict(crop_start_x=w // 10 + 1, crop_start_y=h // 8 + 1, crop_width=w - w // 5 - 2,
                crop_height=h - h // 4 - 2) if case.get("crop") else {}
    return ks.small_pt_params(
        bounces=case["bounces"], render_width=w, render_height=h, spp=spp, spp_prog_interval=spp,
        rng_seed=int(rng.integers(0, 2**31 - 1)), include_background=case.get("background", True),
        backdrop=_BACKDROP, clamp_indirect=case.get("clamp_indirect", 10.0),
        mis_mode=ks.KS_MIS_CONSISTENT if case.get("mis") == "consistent" else ks.KS_MIS_REFERENCE,
        pixel_filter=_FILTERS[case.get("filter", "box")], **crop)


_BATCH_SIZES = [(64, 64), (128, 128), (256, 144), (512, 512), (1024, 576), (1024, 1024)]


def _batch_layout(case):
    """Resolution and spp of each view, fixed by the case; about 40 M paths at most."""
    g = np.random.default_rng(1000 + case["layout"])
    views, paths = [], 0
    for _ in range(case["views"]):
        w, h = _BATCH_SIZES[int(g.integers(len(_BATCH_SIZES)))]
        spp = int(g.choice([4, 16]))
        if paths > 40_000_000:
            w, h, spp = 128, 128, 4
        views.append((w, h, spp))
        paths += w * h * spp
    return views


def _surface_samples(name, n, rng):
    """n points that camera rays see, in the order of the film (as a render records them): position,
    normal, direction to the viewer, and a direction with its weight, cosine-distributed around the normal."""
    hs, sc = _host_scene(name), _scene(name)
    w = max(8, int(math.sqrt(n * 16 / 9)))
    h = max(8, -(-n // w))
    cam = _camera(name, rng, w / h)
    spp = 4
    py, px = np.divmod(np.arange(w * h, dtype=np.int32), np.int32(w))
    rays6 = _device().camera_rays(cam, w, h, spp, 1, px, py, (px + py) % spp)
    rays = np.zeros((w * h, 8), np.float32)
    rays[:, 0:3], rays[:, 4:7], rays[:, 7] = rays6[:, :3], rays6[:, 3:], np.inf
    hits = sc.intersect(rays)
    prim = np.ascontiguousarray(hits[:, 3]).view(np.int32)
    at = np.flatnonzero(prim >= 0)
    at = np.resize(at, n)
    d = torch.from_numpy(rays[at, 4:7]).double()
    tri = torch.from_numpy(hs.vertices[hs.indices[prim[at]].astype(np.int64)]).double()
    nrm = torch.linalg.cross(tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0])
    nrm = nrm / nrm.norm(dim=1, keepdim=True)
    nrm = torch.where((nrm * d).sum(1, keepdim=True) > 0, -nrm, nrm)
    pos = torch.from_numpy(rays[at, 0:3]).double() + d * torch.from_numpy(hits[at, 0:1]).double()
    g = torch.from_numpy(rng.normal(size=(n, 3)))
    wi = nrm + 0.999 * g / g.norm(dim=1, keepdim=True)
    wi = wi / wi.norm(dim=1, keepdim=True)
    weight = torch.from_numpy(rng.exponential(size=n))
    q = torch.cat([pos, nrm, -d], 1)
    return [x.float().contiguous().numpy() for x in (q, wi, weight)]


def _guide_weights(n_grid, n_mlp, rng):
    """Weights of the size training leaves behind: features of 0.1, layers scaled to keep their variance."""
    p = torch.empty(n_grid + n_mlp)
    gen = torch.Generator().manual_seed(int(rng.integers(0, 2**62)))
    p[:n_grid].normal_(0.0, 0.1, generator=gen)
    p[n_grid:].normal_(0.0, 0.2, generator=gen)
    return p.numpy()


def _new_guide(case, **config):
    info = _scene(case["scene"]).info()
    return ks.Guide(_device(), info["bound_lo"], info["bound_hi"], ks.guide_config(**config))


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind, s = case["kind"], _State(case=case, owned=[])
    if kind == "build":
        base = _host_scene(case["scene"])
        moved = base.vertices + rng.normal(scale=2e-3, size=base.vertices.shape).astype(np.float32)
        s["mesh"] = ks.HostScene(moved, base.indices, base.tri_geom, base.geom_material, base.materials, base.lights,
                                 dict(base.camera))
        lo, hi = base.vertices.min(0), base.vertices.max(0)
        rays = np.zeros((case["rays"], 8), np.float32)
        rays[:, 0:3] = rng.uniform(lo - 1, hi + 1, size=(case["rays"], 3))
        d = rng.uniform(lo, hi, size=(case["rays"], 3)) - rays[:, 0:3]
        rays[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
        rays[:, 7] = np.inf
        s["rays"] = rays
        _device()
        return s
    s["scene"] = sc = _scene(case["scene"])
    if kind == "gradient":
        s["guide"] = g = _new_guide(case, log2_table_size=case["log2_table"])
        s["owned"].append(g)
        s["weights"] = _guide_weights(g.n_grid, g.n_mlp, rng)
        g.set_params(s["weights"])
        s["samples"] = _surface_samples(case["scene"], case["samples"], rng)
        return s
    if kind == "batch":
        s["views"] = []
        for w, h, spp in _batch_layout(case):
            view = dict(width=w, height=h, bounces=case["bounces"])
            film = ks.Film(_device(), w, h)
            s["owned"].append(film)
            s["views"].append((_camera(case["scene"], rng, w / h), _params(view, rng, spp), film))
        return s
    s["film"] = film = ks.Film(_device(), case["width"], case["height"], _BACKDROP)
    s["owned"].append(film)
    s["camera"] = _camera(case["scene"], rng, case["width"] / case["height"])
    if kind == "render":
        s["params"] = _params(case, rng, case["spp"])
    else:
        as_guided = dict(case, mis="consistent", clamp_indirect=0.0)
        s["params"] = _params(as_guided, rng, case.get("spp", 1))
    if kind == "guided":
        s["guide"] = g = _new_guide(case, guide_fraction=case["fraction"], max_guided_bounce=case["max_bounce"],
                                    inference_fp8=int(case["fp8"]))
        s["owned"].append(g)
        samples = _surface_samples(case["scene"], 4096, rng)
        g.train_step(*samples)  # a guide samples once it has been trained
        g.set_params(_guide_weights(g.n_grid, g.n_mlp, rng))
        if case["fp8"]:
            g.calibrate_fp8(samples[0])
        g.set_mode(case["fraction"], 0)  # frozen
    if kind == "train":
        s["queries"] = _surface_samples(case["scene"], 4096, rng)[0]
    return s


# ------------------------------------------------------------------------------------------------
# One pass
# ------------------------------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "render":
        state["film"].clear()
        ks.small_pt_render(state["scene"], state["camera"], state["params"], state["film"])
        if case.get("output") == "sums":
            return state["film"].download()
        return state["film"].composite()
    if kind == "batch":
        for _, _, film in state["views"]:
            film.clear()
        ks.small_pt_render_batch(state["scene"], state["views"])
        return [film.composite() for _, _, film in state["views"]]
    if kind == "guided":
        state["film"].clear()
        ks.small_pt_render_guided(state["scene"], state["camera"], state["params"], state["guide"], state["film"])
        return state["film"].composite()
    if kind == "train":
        guide = _new_guide(case, log2_table_size=case["log2_table"], train_spp=1, max_steps_per_pass=case["steps"],
                           seed=1)
        state["film"].clear()
        ks.small_pt_render_guided(state["scene"], state["camera"], state["params"], guide, state["film"])
        out = {"image": state["film"].composite(), "weights": guide.get_params(),
               "mixtures": guide.forward(state["queries"]), "loss": guide.stats()["last_loss"]}
        guide.close()
        return out
    if kind == "gradient":
        loss, grad = state["guide"].gradient(*state["samples"])
        return {"loss": loss, "grad": grad}
    scene = ks.Scene(_device(), state["mesh"], bvh={"builder": 1})
    hits = scene.intersect(state["rays"])
    occluded = scene.occluded(state["rays"])
    scene.close()
    return {"tuv": hits[:, :3], "prim": hits.view(np.int32)[:, 3], "occluded": occluded}


# ------------------------------------------------------------------------------------------------
# What a pass cannot do without
# ------------------------------------------------------------------------------------------------
# closest-hit and shadow rays per path of each scene (the counts of render statistics at the listed sizes)
_RAYS_PER_PATH = {"cornell": (2.90, 2.14), "spheres": (1.27, 0.18), "skymap": (1.34, 0.28), "room": (4.36, 3.27),
                  "foliage": (2.65, 1.84)}
# A ray: ten visits of a node with four child boxes (24 multiply-adds and 24 comparisons each) and four
# watertight triangle tests (about 60 operations each); a path vertex: about 400 operations of light sampling,
# BSDF evaluation, its density and the next direction.
_RAY_FLOPS, _VERTEX_FLOPS = 10 * 4 * 18 + 4 * 60, 400
_MLP_FLOPS = 2 * (39 * 64 + 64 * 64 + 64 * 40)


def _scene_bytes(name):
    hs = _host_scene(name)
    tex = sum(int(np.asarray(t["data"]).nbytes) for t in (hs.textures or []))
    return hs.vertices.nbytes + hs.indices.nbytes + hs.materials.nbytes + tex


def _render_work(scene, paths, pixels, out_bytes):
    c, s = _RAYS_PER_PATH[scene]
    return dict(bytes=_scene_bytes(scene) + 40 * pixels + out_bytes,
                flops=paths * ((c + s) * _RAY_FLOPS + c * _VERTEX_FLOPS))


def work(case):
    kind = case["kind"]
    if kind == "build":
        n = _host_scene(case["scene"]).n_tris
        # mesh in, triangle records and nodes out (48 B and, four to a node, 128 B / 3), rays in, results out;
        # per triangle its box, key and a surface-area comparison per level of a binary tree
        return dict(bytes=_scene_bytes(case["scene"]) + 91 * n + case["rays"] * (32 + 16 + 32 + 1),
                    flops=n * 20 * math.log2(n) + 2 * case["rays"] * _RAY_FLOPS)
    if kind == "gradient":
        n = case["samples"]
        grid = 16 * 2 * 2 ** case["log2_table"]
        # samples in, the features their corners touch, the gradient out; forward, and twice that backward
        return dict(bytes=n * 52 + min(grid * 2, n * 512) + 4 * grid, flops=3 * n * (_MLP_FLOPS + 16 * 8 * 12))
    if kind == "batch":
        views = _batch_layout(case)
        pixels = sum(w * h for w, h, _ in views)
        return _render_work(case["scene"], sum(w * h * spp for w, h, spp in views), pixels, 12 * pixels)
    pixels = case["width"] * case["height"]
    out = 40 * pixels if case.get("output") == "sums" else 12 * pixels
    traced = (case["width"] - case["width"] // 5 - 2) * (case["height"] - case["height"] // 4 - 2) if case.get(
        "crop") else pixels
    paths = traced * case.get("spp", 1)
    c = _render_work(case["scene"], paths, pixels, out)
    if kind == "guided":
        guided = paths * min(_RAYS_PER_PATH[case["scene"]][0], case["max_bounce"] or 99)
        c["flops"] += guided * _MLP_FLOPS
        c["bytes"] += 2 * 16 * 2 * 2**19
    if kind == "train":
        samples = min(case["steps"] * 2**18, 2 * paths)
        c["flops"] += 3 * samples * _MLP_FLOPS
        c["bytes"] += 4 * 4 * 2 * 16 * 2 * 2 ** case["log2_table"]
    return c


# Four times what a camera (or, for the gradient, a query) moved by one unit in the last place changes: every
# float of the pass then rounds another way, and a few paths part at an edge or between two lobes. (largest
# relative error, largest difference of one value) at the samples per pixel of the listed case; the error
# of a mean of fewer samples is larger by the root of their ratio.
_PARTED = {"cornell": (1.5e-4, 0.05, 16), "spheres": (2.5e-3, 0.99, 64), "room": (2e-3, 0.99, 8),
           "foliage": (1.5e-3, 0.35, 16), "skymap": (9e-3, 0.99, 4)}


def tolerance(case):
    kind = case["kind"]
    if kind == "build":  # t, u, v in 32 bits (1e-6 from the 64-bit hits); the same triangles, ties aside
        return {"rel": 4e-6, "max": 1e-3, "differ": 1e-5}
    if kind == "gradient":  # BF16 operands: another rounding of the encoding moves it by 7e-5
        return {"rel": 3e-4, "max": 0.1}
    if kind == "train":  # Adam divides by the gradient's size: near-zero gradients keep only their rounding
        return {"rel": 0.02, "max": 0.99}
    rel, largest, spp = _PARTED[case["scene"]]
    if kind == "guided":  # a mixture's rounding turns every direction drawn from it
        rel *= 2.0 if case["max_bounce"] == 1 else 9.0
    if kind == "batch":
        spp, spp_case = 16, 4
    else:
        spp_case = case["spp"]
    scale = math.sqrt(max(1.0, spp / spp_case))
    return {"rel": min(0.03, rel * scale), "max": min(0.99, largest * scale * scale)}


# ------------------------------------------------------------------------------------------------
# The same in 64 bits
# ------------------------------------------------------------------------------------------------
def exact(case, seed):
    """Ray hits and the guide's gradient in double precision. A render has none: rounding decides now and
    then which of two neighbouring surfaces or lobes a path takes, so a 64-bit render's distance counts the
    paths that parted and says nothing of the arithmetic."""
    if case["kind"] == "build":
        state = prepare(case, seed)
        return {"tuv": _exact_hits(state["mesh"], state["rays"]), "prim": None, "occluded": None}
    if case["kind"] == "gradient":
        state = prepare(case, seed)
        loss, grad = _exact_gradient(state["guide"], state["weights"], *state["samples"])
        return {"loss": loss, "grad": grad}
    return None


def _exact_hits(mesh, rays):
    """Closest hits (t, u, v; -1, 0, 0 for a miss) by testing each ray against every triangle of each
    geometry whose box it meets."""
    cuda = torch.device("cuda")
    r = torch.from_numpy(rays).to(cuda).double()
    o, d = r[:, 0:3], r[:, 4:7]
    vert = torch.from_numpy(mesh.vertices).to(cuda).double()
    tri = vert[torch.from_numpy(mesh.indices.astype(np.int64)).to(cuda)]
    best = torch.full((r.shape[0], 3), -1.0, dtype=torch.float64, device=cuda)
    best[:, 1:] = 0.0
    near = torch.full((r.shape[0],), math.inf, dtype=torch.float64, device=cuda)
    starts = np.flatnonzero(np.diff(mesh.tri_geom.astype(np.int64), prepend=-1))
    for a, b in zip(starts, [*starts[1:], mesh.n_tris]):
        v = tri[int(a):int(b)]
        e1, e2 = v[:, 1] - v[:, 0], v[:, 2] - v[:, 0]
        lo, hi = v.reshape(-1, 3).min(0).values - 1e-6, v.reshape(-1, 3).max(0).values + 1e-6
        t0, t1 = (lo - o) / d, (hi - o) / d
        enter, leave = torch.minimum(t0, t1).amax(1).clamp_min(0), torch.maximum(t0, t1).amin(1)
        rest = torch.nonzero(enter <= leave)[:, 0]
        for part in rest.split(max(1, 2**25 // v.shape[0])):
            D, T = d[part, None, :], o[part, None, :] - v[None, :, 0]
            P, Q = torch.linalg.cross(D, e2[None]), torch.linalg.cross(T, e1[None])
            inv = 1.0 / (e1[None] * P).sum(-1)
            u, w, t = (T * P).sum(-1) * inv, (D * Q).sum(-1) * inv, (e2[None] * Q).sum(-1) * inv
            t = torch.where((u >= 0) & (w >= 0) & (u + w <= 1) & (t > 0), t, math.inf)
            tm, k = t.min(1)
            closer = tm < near[part]
            at, rows = part[closer], torch.nonzero(closer)[:, 0]
            near[at] = tm[closer]
            best[at] = torch.stack([tm[closer], u[rows, k[closer]], w[rows, k[closer]]], 1)
    return best.cpu()


def _exact_gradient(guide, weights, queries, wi, weight):
    """loss = sum of -weight log q(wi) and its gradient: hash-grid features, a 64-64-64-48 ReLU network and
    eight von Mises-Fisher lobes, by autograd."""
    cuda = torch.device("cuda")
    res, lo, inv_ext = guide.grid_info()
    table = guide.n_grid // 32
    p = torch.from_numpy(weights).to(cuda).double().requires_grad_(True)
    q, wi, c = (torch.from_numpy(x).to(cuda).double() for x in (queries, wi, weight))
    total = 0.0
    for part in torch.arange(len(q), device=cuda).split(1 << 16):
        # positions normalised in single precision, as the grid cell of a point is defined
        pos = ((q[part, 0:3].float() - torch.from_numpy(lo).to(cuda)) * torch.from_numpy(inv_ext).to(cuda)).double()
        feats = []
        for level in range(16):
            n = int(res[level])
            x = pos.clamp(0, 1) * n
            cell = x.floor().clamp_max(n - 1)
            f, cell = x - cell, cell.long()
            acc = 0.0
            for corner in range(8):
                off = [(corner >> a) & 1 for a in range(3)]
                i = [cell[:, a] + off[a] for a in range(3)]
                if (n + 1) ** 3 <= table:
                    at = i[0] + (n + 1) * (i[1] + (n + 1) * i[2])
                else:
                    at = (i[0] ^ (i[1] * 2654435761 & 0xFFFFFFFF) ^ (i[2] * 805459861 & 0xFFFFFFFF)) & (table - 1)
                wgt = 1.0
                for a in range(3):
                    wgt = wgt * (f[:, a] if off[a] else 1.0 - f[:, a])
                at = 2 * (at + level * table)
                acc = acc + wgt[:, None] * torch.stack([p[at], p[at + 1]], 1)
            feats.append(acc)
        x = torch.cat([*feats, q[part, 3:9], torch.ones(len(part), 1, dtype=torch.float64, device=cuda)], 1)
        g = guide.n_grid
        w1, w2, w3 = p[g:g + 4096].view(64, 64), p[g + 4096:g + 8192].view(64, 64), p[g + 8192:].view(64, 48)
        out = torch.relu(torch.relu(x @ w1[:39]) @ w2) @ w3
        lobes = out[:, :40].reshape(-1, 8, 5)
        mu = lobes[..., 1:4] / lobes[..., 1:4].norm(dim=-1, keepdim=True)
        kappa = lobes[..., 4].exp().clamp(1e-2, 1e4)
        dirs = wi[part] / wi[part].norm(dim=1, keepdim=True)
        log_norm = kappa.log() - math.log(2 * math.pi) - torch.log(-torch.expm1(-2 * kappa))
        log_lobe = log_norm + kappa * ((mu * dirs[:, None]).sum(-1) - 1).clamp_max(0)
        log_q = torch.logsumexp(torch.log_softmax(lobes[..., 0], 1) + log_lobe, 1)
        loss = -(c[part] * log_q).sum()
        loss.backward()
        total += loss.item()
    return total, p.grad.cpu()
