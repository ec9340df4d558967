"""The sampler's permuted-digit table at its edges: indices of fewer, exactly and one or two more digits than the
ten it looks up (with the eleventh from its permutation byte), whole and half lowest digits, indices of 16
and 17 digits (32 bits and more), sample counts that are no power of two, and dimensions on both sides of
the table's 128. Bit for bit against the oracle's digit loop."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H,spp", [
    (1, 1, 1), (1, 1, 2), (2, 1, 3), (1, 7, 4),  # 0..3 digits
    (512, 3, 1), (512, 512, 2), (512, 300, 4),  # 9, 10
    (1024, 2, 1), (1024, 1024, 2), (1024, 600, 4), (1024, 64, 8),  # 10, 11, 11, 12
    (1920, 1080, 160), (4096, 4096, 256), (8192, 8, 512), (65536, 1, 1), (65536, 2, 2),  # 15, 16, 18, 16, 17
])
def test_table_edges_bit_exact(device, ora, W, H, spp):
    print("sampler table", W, H, spp, flush=True)
    rng = np.random.default_rng(W * 31 + spp)
    n = 64
    px = rng.integers(0, W, n).astype(np.int32)
    py = rng.integers(0, H, n).astype(np.int32)
    s = rng.integers(0, spp, n).astype(np.int32)
    px[0], py[0], s[0] = W - 1, H - 1, spp - 1
    kinds = np.array([2, 1, 2, 1] * 26, np.int32)  # 156 dimensions
    gu, gf = device.sobol_stream(W, H, spp, 11, px, py, s, kinds)
    for i in range(n):
        ou, of = ora.sobol(W, H, spp, 11, int(px[i]), int(py[i]), int(s[i]), kinds)
        assert np.array_equal(gu[i], ou), (i, px[i], py[i], s[i])
        assert np.array_equal(gf[i].view(np.uint32), of.view(np.uint32))
