"""Per-sample radiance of the wavefront against the oracle. Untextured calls of at most 2^16 paths that fit the queue are
carried out by one thread per path; these lists are traced by the kernels that render every larger frame instead: through a
queue that they fill many times over, and as more than 2^16 paths that the queue holds at once. The bars are those of
the same scenes' short lists (test_gpu_parity.py, test_gpu_sky.py, test_gpu_filter.py, test_gpu_configs.py)."""

import numpy as np
import pytest

from test_gpu_sky import SKIES, with_sky

pytestmark = pytest.mark.gpu

# scene, seed, sky map, resolution, spp, bounces, pixel filter, share of samples that agree, share of equal hit flags
CASES = {
    "cornell": ("cornell", 0, None, (256, 256), 16, 8, {}, 0.999, 1.0),
    "cornell_gaussian": ("cornell", 0, None, (128, 128), 16, 8, dict(pixel_filter=1, filter_width=3.0, filter_sigma=0.5),
                         0.999, 1.0),
    "sky_map": ("spheres_small", 1, "z_up_rotated", (256, 256), 16, 8, {}, 0.97, 1.0),
    "spheres": ("spheres", 1, None, (1920, 1080), 64, 12, {}, 0.998, 0.9999),
}


@pytest.mark.parametrize("n,queue", [(20000, 2048), (70000, 0)])
@pytest.mark.parametrize("name", list(CASES))
def test_wavefront_samples_match_oracle(ks, device, ora, name, n, queue):
    print("wavefront samples", name, n, queue, flush=True)
    scene, seed, sky, (W, H), spp, bounces, flt, bar, hit_bar = CASES[name]
    hs = ks.procedural_scene(scene, seed)
    if sky:
        hs = with_sky(ks, hs, SKIES[sky])
    sc = ks.Scene(device, hs)
    osc = ora.OracleScene.from_host_scene(hs)
    rng = np.random.default_rng(n)
    px, py, s = (rng.integers(0, m, n).astype(np.int32) for m in (W, H, spp))
    kw = dict(bounces=bounces, render_width=W, render_height=H, spp=spp, **flt)
    g = sc.trace_samples(hs.camera, ks.small_pt_params(queue_size=queue, **kw), px, py, s)
    o = osc.trace_samples(hs.camera, ora.params(**kw), px, py, s)
    close = np.all(np.abs(g - o) <= 1e-3 * np.maximum(1.0, np.abs(o)), axis=1)
    print("agreement", close.mean(), "hit flags", (g[:, 3] == o[:, 3]).mean(), flush=True)
    assert close.mean() > bar
    assert (g[:, 3] == o[:, 3]).mean() >= hit_bar
    osc.close()
    sc.close()
