"""The grid gradient's accumulation at its edges: batches of one sample, of a wave, of a scatter block and one
more or less, on both sides of the choice between sums in LDS and global atomics, a batch of more than one slice,
the largest tables, and a table whose tiles are so many that every batch is scattered with atomics. Against the
oracle's gradient of the same BF16 operands (bar of test_gpu_guide.py), the slices and the largest tables
against the sum of their parts."""

import ctypes as C

import numpy as np
import pytest

import ks_guide_oracle as go
from test_gpu_guide import BOUNDS, CONFIGS, _params, _queries

pytestmark = pytest.mark.gpu


def _samples(rng, n):
    q = _queries(rng, n, BOUNDS[0], BOUNDS[1])
    wi = rng.standard_normal((n, 3)).astype(np.float32)
    return q, wi, rng.uniform(0.05, 2.0, n).astype(np.float32)


def _check(g, lay, n, seed):
    rng = np.random.default_rng(seed)
    p = _params(g.n_grid, rng)
    g.set_params(p)
    s = _samples(rng, n)
    loss, grad = g.gradient(*s)
    l_ref, g_ref = go.gradient(p, lay, *s, quantised=True)
    assert loss == pytest.approx(l_ref, rel=1e-4)
    o = g.n_grid
    for a, b in ((0, o), (o, o + go.MLP_SIZE)):
        assert np.linalg.norm(grad[a:b] - g_ref[a:b]) < 5e-3 * np.linalg.norm(g_ref[a:b])
    assert np.array_equal(grad[:o] != 0, g_ref[:o] != 0)


# tables of 256 tiles and of some 450 (one and several per level, shared over positions): up to four positions a tile
# are scattered with global atomics, more in LDS
@pytest.mark.parametrize("log2_T,n", [(12, n) for n in (1, 63, 64, 65, 960, 1023, 1024, 1025, 4097)]
                         + [(15, n) for n in (1, 63, 64, 65, 1023, 1024, 1025, 1600, 2047, 2049, 4097)])
def test_batch_edges(ks, device, n, log2_T):
    print("scatter", n, log2_T, flush=True)
    cfg = dict(CONFIGS["small"], log2_table_size=log2_T)
    g = ks.Guide(device, *BOUNDS, ks.guide_config(seed=7, **cfg))
    _check(g, go.Layout(log2_T, 4.0, 256.0, *BOUNDS), n, n)
    g.close()


def test_large_table_uses_atomics(ks, device):
    """Sixteen hashed levels of 2^22 entries: 4096 tiles."""
    print("scatter atomics", flush=True)
    g = ks.Guide(device, *BOUNDS, ks.guide_config(seed=7, log2_table_size=22, base_resolution=256.0, max_resolution=512.0))
    _check(g, go.Layout(22, 256.0, 512.0, *BOUNDS), 130, 5)
    g.close()


def test_large_default_table_in_lds(ks, device):
    """2^22 entries at the default resolutions: 1722 tiles, in LDS from 6888 positions on."""
    print("scatter 2^22 in LDS", flush=True)
    g = ks.Guide(device, *BOUNDS, ks.guide_config(seed=7, log2_table_size=22))
    _check(g, go.Layout(22, 16.0, 256.0, *BOUNDS), 8192, 6)
    g.close()


@pytest.mark.parametrize("log2_T,tiles", [(23, 2317), (24, 2907)])
def test_large_default_tables_agree_with_atomics(ks, device, log2_T, tiles):
    """A batch of more than four positions a tile, scattered in LDS, against its halves, scattered with atomics: the
    same FP32 terms in another order. An entry of m terms errs by about sqrt(m) 2^-24 of their absolute sum (27 of the
    coarsest level's, 14 000 of a weight's: 8e-6), with an allowance of 4 for cancellation between them."""
    print("scatter", log2_T, flush=True)
    n = 4 * tiles // 64 * 64 + 128
    g = ks.Guide(device, *BOUNDS, ks.guide_config(seed=7, log2_table_size=log2_T))
    q, wi, c = _samples(np.random.default_rng(log2_T), n)
    loss, grad = g.gradient(q, wi, c)
    k = n // 2
    l0, want = g.gradient(q[:k], wi[:k], c[:k])
    l1, part = g.gradient(q[k:], wi[k:], c[k:])
    g.close()
    want += part
    assert loss == pytest.approx(l0 + l1, rel=1e-9)
    o = len(grad) - go.MLP_SIZE
    for a, b in ((0, o), (o, o + go.MLP_SIZE)):
        err = np.linalg.norm(grad[a:b] - want[a:b]) / np.linalg.norm(want[a:b])
        print("relative L2 difference", err, flush=True)
        assert err < 3.2e-5
    # no entry is lost or touched by one of them alone
    assert np.count_nonzero(grad[:o]) == np.count_nonzero(want[:o])


def test_slices_add_up(ks, device):
    """2^20 + 130 samples are two slices. Each entry's sum of m FP32 terms errs by at most m 2^-24 of the terms'
    absolute sum, about sqrt(m) 2^-24 when rounding errors are independent: below 1e-4 for the 2^20 terms that
    meet in a weight, with an allowance of 4 for cancellation between them."""
    print("scatter slices", flush=True)
    g = ks.Guide(device, *BOUNDS, ks.guide_config(seed=7, **CONFIGS["small"]))
    rng = np.random.default_rng(9)
    g.set_params(_params(g.n_grid, rng))
    q, wi, c = _samples(rng, (1 << 20) + 130)
    k = 1 << 20
    l0, g0 = g.gradient(q[:k], wi[:k], c[:k])
    l1, g1 = g.gradient(q[k:], wi[k:], c[k:])
    loss, grad = g.gradient(q, wi, c)
    assert loss == pytest.approx(l0 + l1, rel=1e-9)
    o = g.n_grid
    for a, b in ((0, o), (o, o + go.MLP_SIZE)):
        want = g0[a:b].astype(np.float64) + g1[a:b]
        err = np.linalg.norm(grad[a:b] - want) / np.linalg.norm(want)
        print("relative L2 difference", err, flush=True)
        assert err < 4e-4
    g.close()


@pytest.mark.parametrize("res", [15, 16, 255, 256, 4194303])
def test_dense_and_hashed_levels(ks, device, res):
    """Resolutions at which a level stops being dense ((15 + 1)^3 entries are the table's), and whose cube leaves 32 and
    64 bits ((4194303 + 1)^3 = 2^66). With zero grid features the features' gradient does not depend on the
    corners' weights, which sum to one: every level of the table holds the same sums as the oracle's, whatever the
    rounding of a position inside so fine a cell. Bar: that of the gradients."""
    print("levels", res, flush=True)
    g = ks.Guide(device, *BOUNDS, ks.guide_config(seed=7, log2_table_size=12, base_resolution=float(res),
                                                  max_resolution=float(res)))
    assert g.grid_info()[0].tolist() == [res] * go.LEVELS
    rng = np.random.default_rng(res % 1000)
    p = _params(g.n_grid, rng)
    p[: g.n_grid] = 0
    g.set_params(p)
    s = _samples(rng, 1500)
    _, grad = g.gradient(*s)
    lay = go.Layout(12, float(res), float(res), *BOUNDS)
    _, g_ref = go.gradient(p, lay, *s, quantised=True)
    a, b = (x[: g.n_grid].reshape(go.LEVELS, -1, go.FEATURES).sum(axis=1, dtype=np.float64) for x in (grad, g_ref))
    assert np.linalg.norm(a - b) < 5e-3 * np.linalg.norm(b)
    o = g.n_grid
    assert np.linalg.norm(grad[o:] - g_ref[o:]) < 5e-3 * np.linalg.norm(g_ref[o:])
    if res < 1000:
        assert np.linalg.norm(grad[:o] - g_ref[:o]) < 5e-3 * np.linalg.norm(g_ref[:o])
    assert np.isfinite(g.forward(s[0])).all()
    g.close()


@pytest.mark.parametrize("res", [4294967296.0, float("inf"), float("nan")])
def test_resolutions_beyond_32_bits_are_refused(ks, device, res):
    with pytest.raises(ks.KsError) as e:
        ks.Guide(device, *BOUNDS, ks.guide_config(max_resolution=res))
    assert e.value.status == ks.KS_ERR_INVALID


def test_guides_share_the_training_scratch(ks, device):
    """A second guide's first step takes memory for its samples (64 B each) and weight partials (768 waves x 11264
    floats) alone: the rows, positions and gradients between the kernels lie in the device's scratch. Steps by turns
    give what each guide's own steps give."""
    lib = ks.load_library()

    def free():
        f, t = C.c_size_t(), C.c_size_t()
        assert lib.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    n = 1 << 18
    rng = np.random.default_rng(4)
    s = [_samples(rng, m) for m in (n, 5000)]
    g = [ks.Guide(device, *BOUNDS, ks.guide_config(seed=k, **CONFIGS["small"])) for k in (1, 2)]
    alone = [x.gradient(*b) for x in g[:1] for b in s]
    before = free()
    turns = []
    for b in s:
        turns.append((g[1].gradient(*b), g[0].gradient(*b)))
    took = before - free()
    print("the second guide took", took, flush=True)
    assert took < 64 * n + 4 * 768 * 11264 + (8 << 20)
    for (l0, g0), (_, (l1, g1)) in zip(alone, turns):
        assert l0 == pytest.approx(l1, rel=1e-9)
        assert np.linalg.norm(g0 - g1) < 1e-4 * np.linalg.norm(g0)
    for x in g:
        x.close()
