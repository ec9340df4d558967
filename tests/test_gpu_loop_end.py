"""The wavefront loop's end: known from the bounce count where the queue holds the whole pass, read from the
control block otherwise, and a batch that leaves graph replay for bounded launches. Every path must be
carried to its end in each, so the films are equal bit for bit. Passes of at most 2^16 paths that fit their queue
are carried out by one thread per path instead, so only the largest size here has a known end."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bounces", [0, 1, 2, 7, 8, 17])
@pytest.mark.parametrize("size,spp", [((3, 1), 1), ((31, 17), 3), ((64, 48), 4), ((331, 199), 1)])
def test_known_and_read_ends_agree(ks, device, cornell, bounces, size, spp):
    print("loop end", bounces, size, spp, flush=True)
    sc = ks.Scene(device, cornell)
    w, h = size
    out = []
    # the queue that holds every path; one that refills (at least 256 slots); batches, replayed and eager
    for queue, batch, graph in ((0, False, False), (256, False, False), (256, True, True), (4096, True, True),
                                (0x10000, True, False)):
        film = ks.Film(device, w, h)
        p = ks.small_pt_params(bounces=bounces, render_width=w, render_height=h, spp=spp, spp_prog_interval=spp,
                               rng_seed=7, queue_size=queue)
        if batch:
            st = ks.small_pt_render_batch(sc, [(cornell.camera, p, film)], queue_size=queue, graph=graph)
        else:
            st = ks.small_pt_render(sc, cornell.camera, p, film)
        out.append((film.download(), st["rays_closest"], st["rays_shadow"]))
        n = w * h * spp
        if n <= 1 << 16 and n <= max(queue, 256 if queue else n):
            assert st["iterations"] == 1  # one thread per path
        elif queue == 0:  # known end: one iteration per vertex of the longest path, unless a read found none left
            assert st["iterations"] == bounces + 1 or (bounces > 8 and 8 < st["iterations"] <= bounces)
        else:
            assert st["iterations"] >= n // queue + bool(n % queue)
        film.close()
    sc.close()
    (rgb, wts), rc, rs = out[0]
    assert wts.sum() == w * h * spp
    for (r, g), c, s in out[1:]:
        assert np.array_equal(r, rgb) and np.array_equal(g, wts) and (c, s) == (rc, rs)


@pytest.mark.parametrize("name,seed", [("cornell", 0), ("spheres_small", 1)])
@pytest.mark.parametrize("w,h,spp", [(64, 1, 1), (65, 1, 1), (512, 128, 1), (331, 99, 2), (331, 33, 5), (513, 128, 1)])
def test_whole_paths_equal_the_wavefront(ks, device, name, seed, w, h, spp):
    """Up to 2^16 paths, one thread per path; just above, and with a queue that cannot hold them, the wavefront."""
    print("whole paths", name, w, h, spp, flush=True)
    hs = ks.procedural_scene(name, seed)
    sc = ks.Scene(device, hs)
    cam = dict(hs.camera)
    cam["aspect"] = w / h
    out = []
    for queue in (0, max(256, w * h * spp // 3)):
        film = ks.Film(device, w, h)
        p = ks.small_pt_params(bounces=9, render_width=w, render_height=h, spp=spp, spp_prog_interval=spp, rng_seed=3,
                               queue_size=queue)
        st = ks.small_pt_render(sc, cam, p, film)
        out.append((film.download(), st))
        film.close()
    sc.close()
    ((a, wa), sa), ((b, wb), sb) = out
    print("iterations", sa["iterations"], sb["iterations"], flush=True)
    assert np.array_equal(a, b) and np.array_equal(wa, wb)
    for k in ("rays_closest", "rays_shadow", "rays_tail", "paths", "nonfinite"):
        assert sa[k] == sb[k], k


@pytest.mark.parametrize("w,h,spp,bounces,whole", [(128, 128, 1, 2, True), (256, 128, 1, 2, False), (64, 64, 16, 7, True),
                                                   (64, 64, 16, 6, False), (32, 32, 1, 1, False), (9, 7, 1, 2, True)])
def test_large_scenes_take_whole_paths_where_bounces_pay(ks, device, w, h, spp, bounces, whole):
    """1.31 M triangles, 2 doublings of 2^18: 49152 (bounces - 1) against twice the paths, those of several samples a
    pixel counted double. Either way, and in a batch, the film is that of a queue too small for whole paths."""
    print("bounces that pay", w, h, spp, bounces, flush=True)
    hs = ks.procedural_scene("spheres", 1)
    sc = ks.Scene(device, hs, bvh={"builder": 1})
    cam = dict(hs.camera)
    cam["aspect"] = w / h
    out = []
    for queue, batch in ((0, False), (max(256, w * h * spp - 1), False), (0, True)):
        film = ks.Film(device, w, h)
        p = ks.small_pt_params(bounces=bounces, render_width=w, render_height=h, spp=spp, spp_prog_interval=spp,
                               queue_size=queue)
        if batch:
            st = ks.small_pt_render_batch(sc, [(cam, p, film)])
        else:
            st = ks.small_pt_render(sc, cam, p, film)
        out.append((film.download(), st))
        film.close()
    sc.close()
    for (rgb, wts), st in out[::2]:
        assert (st["launches"]["tail"] == 1) == whole
        assert np.array_equal(rgb, out[1][0][0]) and np.array_equal(wts, out[1][0][1])
        assert st["rays_closest"] == out[1][1]["rays_closest"] and st["rays_shadow"] == out[1][1]["rays_shadow"]
