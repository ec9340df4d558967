"""The traversal's opacity test for every way a field can be read: constant, nearest, bilinear and cubic samplers,
u8 / u16 / f32 textures in both colour spaces, a swizzle to each channel and to none, both wrap modes, uv
transform, flip and scale. Rays through stacks of alpha-tested quads meet the same triangles as the
oracle's, closest and any hit. Opacities are a function of the hit; a ray within rounding of a texel border or
of its own hash may part, so 99.9% must agree."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def scene(api, sampler, dtype, srgb, channels, swizzle, wrap):
    rng = np.random.default_rng(17)
    v, tc, idx, tg = [], [], [], []
    for k in range(12):
        z = 0.1 * k
        b = len(v)
        v += [(0, 0, z), (1, 0, z), (1, 1, z), (0, 1, z)]
        tc += [(-0.3, 0.2), (1.7, 0.1), (1.9, 2.1), (-0.1, 1.8)]
        idx += [[b, b + 1, b + 2], [b, b + 2, b + 3]]
        tg += [k, k]
    data = rng.integers(0, 256, (9, 13, channels)) / 255.0
    data = data.astype(np.float32) if dtype == "f32" else np.round(
        data * (255 if dtype == "u8" else 65535)).astype(np.uint8 if dtype == "u8" else np.uint16)
    mats = np.zeros(2, api.MATERIAL_DTYPE)
    mats["basecolor"], mats["roughness"], mats["ior"], mats["specular_r0_mul"] = 0.5, 0.6, 1.5, 0.5
    f = api.field_desc
    tex = f(value=0.4) if sampler is None else f(
        texture=0, sampler=sampler, cubic_kernel=api.KS_CUBIC_MITCHELL, swizzle=(swizzle,), wrap_u=wrap, wrap_v=wrap,
        uv_scale=(1.3, 0.7), uv_offset=(0.1, -0.2), scale=(0.9,), flip_v=wrap == api.KS_WRAP_REPEAT)
    fields = {0: api.material_fields(mats[0], opacity=tex)}
    return api.HostScene(
        vertices=np.asarray(v, np.float32), indices=np.asarray(idx, np.uint32), tri_geom=np.asarray(tg, np.uint32),
        geom_material=np.asarray([0] * 11 + [1], np.uint32), materials=mats, lights=np.zeros(0, api.LIGHT_DTYPE),
        camera=dict(pos=(0.5, 0.5, 3), target=(0.5, 0.5, 0), up=(0, 1, 0), vfov=40.0, aspect=1.0),
        texcoords=np.asarray(tc, np.float32),
        textures=[dict(data=data, srgb=srgb, mipmaps=False)], material_fields=fields)


CASES = [(None, "u8", False, 1, 0, 0)]
CASES += [(s, d, g, c, w, r) for s, d, g, c, w, r in [
    (0, "u8", False, 1, 0, 0), (0, "u8", True, 4, 3, 1), (0, "u16", False, 2, 1, 0), (0, "f32", False, 3, 2, 1),
    (1, "u8", False, 3, 2, 1), (1, "u16", True, 4, 0, 0), (1, "f32", False, 1, 0, 1), (2, "u8", True, 1, 0, 0),
    (2, "u16", False, 4, 3, 1), (2, "f32", True, 2, 1, 0), (3, "u8", False, 4, 1, 0), (0, "u8", False, 3, -1, 0)]]


@pytest.mark.parametrize("sampler,dtype,srgb,channels,swizzle,wrap", CASES)
def test_opacity_fields_match_oracle(ks, device, ora, sampler, dtype, srgb, channels, swizzle, wrap):
    print("opacity", sampler, dtype, srgb, channels, swizzle, wrap, flush=True)
    hs = scene(ks, sampler, dtype, srgb, channels, swizzle, wrap)
    sc = ks.Scene(device, hs)
    osc = ora.OracleScene.from_host_scene(hs)
    rng = np.random.default_rng(3)
    n = 20000
    o = np.stack([rng.uniform(0, 1, n), rng.uniform(0, 1, n), np.where(np.arange(n) % 2 == 0, 3.0, -2.0)], -1)
    t = np.stack([rng.uniform(0, 1, n), rng.uniform(0, 1, n), rng.uniform(0, 1.1, n)], -1)
    d = (t - o) / np.linalg.norm(t - o, axis=1, keepdims=True)
    rays = np.zeros((n, 8), np.float32)
    rays[:, 0:3], rays[:, 4:7], rays[:, 7] = o, d, 100.0
    g, r = sc.intersect(rays)[:, 3].view(np.int32), osc.intersect(rays)[:, 3].view(np.int32)
    print("agree", (g == r).mean(), "hit", (r >= 0).mean(), flush=True)
    assert (g == r).mean() > 0.999
    assert (sc.occluded(rays).astype(bool) == (g >= 0)).mean() > 0.999
    sc.close()


@pytest.mark.parametrize("w,h,spp", [(63, 1, 1), (97, 61, 3), (500, 300, 8)])
@pytest.mark.parametrize("branching", [4, 2])
def test_ray_replacement_does_not_change_a_render(ks, device, w, h, spp, branching):
    """Alpha-tested path launches mix camera rays, which stay together, with later rays, which are replaced at
    once; the mix and the lane a ray falls to depend on the queue. The films and ray counts must not."""
    print("replacement", w, h, spp, branching, flush=True)
    import sys
    from pathlib import Path

    sys.path.insert(0, str(Path(__file__).parent))
    from texture_scenes import textured_box

    hs = textured_box()
    sc = ks.Scene(device, hs, bvh={"branching": branching})
    cam = dict(hs.camera)
    cam["aspect"] = w / h
    out = []
    for queue in (0, 256 if w * h * spp < 20000 else 65536, max(256, w * h * spp * 2 // 3)):
        film = ks.Film(device, w, h)
        p = ks.small_pt_params(bounces=7, render_width=w, render_height=h, spp=spp, spp_prog_interval=spp,
                               rng_seed=5, queue_size=queue)
        st = ks.small_pt_render(sc, cam, p, film)
        out.append((film.download(), st))
        film.close()
    sc.close()
    (a, wa), sa = out[0]
    for (b, wb), sb in out[1:]:
        assert np.array_equal(a, b) and np.array_equal(wa, wb)
        for k in ("rays_closest", "rays_shadow", "paths", "nonfinite"):
            assert sa[k] == sb[k], k
