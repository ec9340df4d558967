"""ks_film_composite on the device against the FP64 formula on the downloaded sums (RenderTarget2::composite,
render_target.cpp:187-192, lerp with a float t): equal bit for bit, for films with hits, misses and pixels no
sample reached, of one pixel, of a block of pixels and one more, and after the film was cleared."""

import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def expected(rgb, w, backdrop):
    hit, total = w[..., 0], (w[..., 0] + w[..., 1]).astype(np.uint32)
    t = np.where(total == 0, 0.0, hit / np.maximum(total, 1)).astype(np.float32)
    fg = np.where(hit[..., None] == 0, 0.0, rgb / np.maximum(hit, 1)[..., None])
    one_minus = (np.float32(1) - t).astype(np.float64)[..., None]
    return (one_minus * np.asarray(backdrop, np.float32).astype(np.float64) + t.astype(np.float64)[..., None] * fg).astype(
        np.float32)


# the last two: 2^21 pixels, one part of the device's buffer, and 3073 more
@pytest.mark.parametrize("w,h", [(1, 1), (256, 1), (257, 1), (53, 41), (2048, 1024), (2049, 1025)])
@pytest.mark.parametrize("crop", [False, True])
def test_composite_matches_formula(ks, device, spheres_small, w, h, crop):
    print("composite", w, h, crop, flush=True)
    backdrop = (0.3, 0.1, 0.7)
    sc = ks.Scene(device, spheres_small)
    film = ks.Film(device, w, h, backdrop)
    cam = dict(spheres_small.camera)
    cam["aspect"] = w / h
    kw = dict(crop_start_x=w // 3, crop_start_y=h // 3, crop_width=max(1, w // 2), crop_height=max(1, h // 2)) if crop else {}
    p = ks.small_pt_params(bounces=3, render_width=w, render_height=h, spp=5, spp_prog_interval=5,
                           include_background=False, **kw)
    for clear in (False, True):
        if clear:
            film.clear()
        else:
            ks.small_pt_render(sc, cam, p, film)
        rgb, wts = film.download()
        got = film.composite()
        assert np.array_equal(got.view(np.uint32), expected(rgb, wts, backdrop).view(np.uint32))
    film.close()
    sc.close()


def test_composite_takes_no_device_memory(ks, device):
    """A film can be composited however little device memory is free, and holds none for it afterwards."""
    lib = ks.load_library()

    def free():
        f, t = C.c_size_t(), C.c_size_t()
        assert lib.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    films = [ks.Film(device, 1920, 1080) for _ in range(4)]
    before = free()
    for f in films:
        f.composite()
    print("taken by four composites", before - free(), flush=True)
    assert free() == before
    for f in films:
        f.close()
