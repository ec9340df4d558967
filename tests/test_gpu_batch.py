"""Batched renders (ks_small_pt_render_batch): many views of one scene in one wavefront. Every view's film
must equal, bit for bit, the film of that view rendered alone: the same Sobol samples per pixel, folded
in the same order. Covered: mixed resolutions, spp (including non powers of two), seeds, a crop and a
moved camera; graph replay and eager launches; the autotuner and a fixed queue."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _views(ks, cornell):
    cam2 = dict(cornell.camera)
    cam2["pos"] = (0.2, 0.6, 2.0)
    specs = [
        (cornell.camera, dict(render_width=64, render_height=64, spp=4, rng_seed=0)),
        (cornell.camera, dict(render_width=128, render_height=72, spp=16, rng_seed=3)),
        (cam2, dict(render_width=96, render_height=96, spp=5, rng_seed=1)),
        (cornell.camera, dict(render_width=200, render_height=120, spp=8, rng_seed=2, crop_start_x=20,
                              crop_start_y=10, crop_width=100, crop_height=50)),
        (cam2, dict(render_width=32, render_height=48, spp=64, rng_seed=7)),
    ]
    out = []
    for cam, kw in specs:
        p = ks.small_pt_params(bounces=12, spp_prog_interval=kw["spp"], **kw)
        out.append((cam, p, kw))
    return out


@pytest.mark.parametrize("mode", ["graph_autotune", "eager_fixed"])
def test_batch_equals_single_views(ks, device, cornell, mode):
    sc = ks.Scene(device, cornell)
    views = _views(ks, cornell)
    films = [ks.Film(device, kw["render_width"], kw["render_height"]) for _, _, kw in views]
    if mode == "graph_autotune":
        st = ks.small_pt_render_batch(sc, [(c, p, f) for (c, p, _), f in zip(views, films)])
    else:
        st = ks.small_pt_render_batch(sc, [(c, p, f) for (c, p, _), f in zip(views, films)], queue_size=1 << 14,
                                      trace_blocks_per_cu=4, graph=False)
    print(mode, "queue", st["queue_size"], "blocks/CU", st["trace_blocks_per_cu"], "paths", st["paths"],
          "iterations", st["iterations"], flush=True)
    assert st["paths"] == sum(kw["spp"] * (kw.get("crop_width") or kw["render_width"]) *
                              (kw.get("crop_height") or kw["render_height"]) for _, _, kw in views)
    for (cam, p, kw), f in zip(views, films):
        alone = ks.Film(device, kw["render_width"], kw["render_height"])
        ks.small_pt_render(sc, cam, p, alone)
        a, wa = f.download()
        b, wb = alone.download()
        assert np.array_equal(wa, wb), kw
        assert np.array_equal(a, b), kw
        alone.close()
    for f in films:
        f.close()
    sc.close()


@pytest.mark.parametrize("graph,queue,scale", [(True, 0, 4), (True, 1 << 13, 1), (True, 0, 1), (False, 1 << 13, 1)])
def test_views_split_across_chunks(ks, device, cornell, graph, queue, scale):
    """A small chunk budget (50 000 items) splits the batch into four chunks, and the spp of the first
    three views across chunk boundaries (segments starting at s0 > 0, one sentinel per chunk): every film
    still equals its single render bit for bit. At four times the samples and the budget the chunks exceed 2^16 items
    and the autotuner's probe runs on the first chunk's partial segment list; with a queue smaller than them
    the chunks are replayed graphs or eager launches; else each is carried out by one thread per path."""
    sc = ks.Scene(device, cornell)
    cam2 = dict(cornell.camera)
    cam2["pos"] = (0.3, 0.4, 2.2)
    specs = [(cornell.camera, dict(render_width=64, render_height=64, spp=16, rng_seed=1)),
             (cam2, dict(render_width=32, render_height=32, spp=64, rng_seed=2)),
             (cornell.camera, dict(render_width=48, render_height=40, spp=9, rng_seed=3))]
    for _, kw in specs:
        kw["spp"] *= scale
    views = [(cam, ks.small_pt_params(bounces=12, spp_prog_interval=kw["spp"], **kw), kw) for cam, kw in specs]
    films = [ks.Film(device, kw["render_width"], kw["render_height"]) for _, _, kw in views]
    kwargs = dict(max_chunk_items=50_000 * scale, graph=graph)
    if queue:
        kwargs.update(queue_size=queue, trace_blocks_per_cu=4)
    st = ks.small_pt_render_batch(sc, [(c, p, f) for (c, p, _), f in zip(views, films)], **kwargs)
    print("chunks", st["batch_chunks"], "queue", st["queue_size"], "iterations", st["iterations"], flush=True)
    assert st["batch_chunks"] == (4 if scale == 1 else 3)
    if queue or scale > 1:
        assert st["iterations"] >= 8 * st["batch_chunks"]
    else:
        assert st["iterations"] == 4
    for (cam, p, kw), f in zip(views, films):
        alone = ks.Film(device, kw["render_width"], kw["render_height"])
        ks.small_pt_render(sc, cam, p, alone)
        a, wa = f.download()
        b, wb = alone.download()
        assert np.array_equal(wa, wb) and np.array_equal(a, b), kw
        alone.close()
    for f in films:
        f.close()
    sc.close()


def test_batch_folds_every_remainder_of_eight(ks, device, cornell):
    """The film fold reads eight samples of a pixel at a time, then the rest one by one."""
    sc = ks.Scene(device, cornell)
    views = [ks.small_pt_params(bounces=4, render_width=37, render_height=5, spp=n, spp_prog_interval=n, rng_seed=n)
             for n in (1, 7, 8, 9, 15, 16, 17, 23)]
    films = [ks.Film(device, 37, 5) for _ in views]
    ks.small_pt_render_batch(sc, [(cornell.camera, p, f) for p, f in zip(views, films)])
    for p, f in zip(views, films):
        alone = ks.Film(device, 37, 5)
        ks.small_pt_render(sc, cornell.camera, p, alone)
        a, wa = f.download()
        b, wb = alone.download()
        alone.close()
        f.close()
        assert np.array_equal(a, b) and np.array_equal(wa, wb)
    sc.close()


def test_small_batches_are_not_tuned(ks, device, cornell):
    """Queue size and traversal blocks are the wavefront's settings: a batch carried out by one thread per path is
    not timed over them and reports the defaults, whichever probe would have been the fastest. Chunks of both
    kinds in one batch give the films of single renders."""
    sc = ks.Scene(device, cornell)
    for n in range(1, 9):
        film = ks.Film(device, 32, 32)
        p = ks.small_pt_params(bounces=4, render_width=32, render_height=32, spp=n, spp_prog_interval=n)
        st = ks.small_pt_render_batch(sc, [(cornell.camera, p, film)])
        assert (st["iterations"], st["queue_size"], st["trace_blocks_per_cu"]) == (1, 1024 * n, 8)
        film.close()
    sizes = [(32, 32, 4), (512, 384, 1), (40, 20, 3)]  # chunks of 4096, 196 608 and 2400 items
    films = [ks.Film(device, w, h) for w, h, _ in sizes]
    params = [ks.small_pt_params(bounces=4, render_width=w, render_height=h, spp=n, spp_prog_interval=n)
              for w, h, n in sizes]
    st = ks.small_pt_render_batch(sc, [(cornell.camera, p, f) for p, f in zip(params, films)], max_chunk_items=197_000)
    print("chunks", st["batch_chunks"], "iterations", st["iterations"], "queue", st["queue_size"], flush=True)
    assert st["batch_chunks"] == 3 and st["iterations"] > 5
    for p, f in zip(params, films):
        alone = ks.Film(device, f.width, f.height)
        ks.small_pt_render(sc, cornell.camera, p, alone)
        assert all(np.array_equal(a, b) for a, b in zip(f.download(), alone.download()))
        alone.close()
        f.close()
    sc.close()


@pytest.mark.parametrize("queue", [1 << 13, 1 << 17])
def test_kernel_times_of_a_graph_batch_are_none_or_whole(ks, device, cornell, queue):
    """Replayed iterations record no events, so no iteration of a graph batch does, nor its small last chunk (9600
    items, one thread per path); eagerly launched, every class that ran is timed."""
    sc = ks.Scene(device, cornell)
    film = ks.Film(device, 160, 120)
    p = ks.small_pt_params(bounces=8, render_width=160, render_height=120, spp=8, spp_prog_interval=8)
    small = ks.Film(device, 160, 60)
    q = ks.small_pt_params(bounces=8, render_width=160, render_height=60, spp=1, spp_prog_interval=1)
    device.set_timing(True)
    st = {g: ks.small_pt_render_batch(sc, [(cornell.camera, p, film), (cornell.camera, q, small)], queue_size=queue,
                                      graph=g, max_chunk_items=160 * 120 * 8) for g in (True, False)}
    device.set_timing(False)
    film.close()
    small.close()
    sc.close()
    print(queue, st[True]["kernel_ms"], st[True]["launches"], st[False]["kernel_ms"], flush=True)
    for k in ("raygen", "closest", "shade"):
        assert st[True]["kernel_ms"][k] == 0 and st[True]["launches"][k] == 0
        assert st[False]["kernel_ms"][k] > 0 and st[False]["launches"][k] > 0
    assert st[True]["kernel_ms"]["film"] > 0 and st[True]["batch_chunks"] == 2
