"""The radiance cache's encoder, network and gradient scatter at the record counts where their waves, tiles and
workgroups end."""
import numpy as np
import pytest

import test_gpu_rc as base
import vierkant_amd as vk

pytestmark = pytest.mark.gpu

# 16-record tiles, 32 record pairs a wave, 64 training samples, 128 encoded and 256 queried records a workgroup
SIZES = [1, 15, 16, 17, 31, 33, 63, 65, 127, 128, 129, 255, 257, 513]


@pytest.fixture()
def cache(ctx):
    c = vk.RadianceCache(ctx, vk.default_rc_params(log2_table=base.LOG2_T), seed=1)
    c.set_bounds(base.BMIN, base.BMAX)
    rng = np.random.default_rng(9)
    c.set_params(rng.normal(scale=0.2, size=c.n_mlp).astype(np.float32),
                 rng.uniform(-0.5, 0.5, size=(16, 1 << base.LOG2_T, 2)).astype(np.float32))
    yield c
    c.close()


def test_queries_do_not_depend_on_the_batch(cache):
    """a record's prediction is the same bits in a batch of any size (1,024 records: the whole-tile case that
    test_gpu_rc compares with the numpy restatement)"""
    rec = base.world_records(1024, 21)
    want = cache.query(rec)
    assert np.any(want != 0)
    for n in SIZES:
        assert np.array_equal(cache.query(rec[:n]), want[:n]), n


@pytest.mark.parametrize("n", SIZES)
def test_gradients_at_tile_edges(cache, n):
    """against the numpy restatement: only its entries are touched, and values agree to 12 roundings to bfloat16 (6
    layers forward, 6 back, 2^-8 each: 4.7 %) of the largest one"""
    rec = base.world_records(n, 22)
    tg = np.random.default_rng(23).uniform(0, 2, (n, 3)).astype(np.float32)
    cache.train(rec, tg, grad_only=True)
    g_mlp, g_grid = cache.get_gradients()
    mlp, grid = cache.get_params()
    _, w_mlp, w_grid = base.R.train_gradients(rec, tg, base.stored_grid(grid), mlp, base.BMIN, base.inv_extent())
    assert not np.any((g_grid != 0) & (w_grid == 0))
    assert np.abs(g_grid - w_grid).max() <= 0.047 * np.abs(w_grid).max()
    assert np.abs(g_mlp - w_mlp).max() <= 0.047 * np.abs(w_mlp).max()
