"""The radiance cache's encoder, network and gradient scatter at the record counts where their waves, tiles and
workgroups end."""
import ctypes

import numpy as np
import pytest
import torch

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
    layers forward, 6 back, 2^-8 each: 4.7 %) of the largest one; entries that only the last record, the one at the
    tile's edge, touches agree to as much of that record's largest"""
    rec = base.world_records(n, 22)
    tg = np.random.default_rng(23).uniform(0, 2, (n, 3)).astype(np.float32)
    cache.train(rec, tg, grad_only=True)
    g_mlp, g_grid = cache.get_gradients()
    mlp, grid = cache.get_params()
    _, w_mlp, w_grid = base.R.train_gradients(rec, tg, base.stored_grid(grid), mlp, base.BMIN, base.inv_extent())
    assert not np.any((g_grid != 0) & (w_grid == 0))
    assert np.abs(g_grid - w_grid).max() <= 0.047 * np.abs(w_grid).max()
    assert np.abs(g_mlp - w_mlp).max() <= 0.047 * np.abs(w_mlp).max()


QUERY_PASS, TRAIN_PASS = 1 << 20, 1 << 16  # records that one pass over the encoder's buffers takes


def test_queries_of_several_passes(cache):
    """past the records that the encoder's buffers hold, a query goes on from their start"""
    rec = base.world_records(5000, 24)
    want = cache.query(rec)
    n = 2 * QUERY_PASS + 129
    got = cache.query(np.tile(rec, (n // len(rec) + 1, 1))[:n])
    assert np.array_equal(got, np.tile(want, (n // len(want) + 1, 1))[:n])


def test_training_over_several_passes(cache):
    """four passes' records, the first pass's four times over: the mean over all is the mean over one pass, and every
    factor but the power of two 1 / n the same, so only the order of the sums differs (2^-24 times the 4,096
    additions of a weight's partial sums at most; the table's in binary16 with its 2^-11 per addition, hundreds
    of them for a coarse entry)"""
    rec = base.world_records(TRAIN_PASS, 25)
    tg = np.random.default_rng(26).uniform(0, 2, (TRAIN_PASS, 3)).astype(np.float32)
    got = []
    for k in (1, 4):
        loss = cache.train(np.tile(rec, (k, 1)), np.tile(tg, (k, 1)), grad_only=True)
        got.append((loss, *cache.get_gradients()))
    (l1, m1, g1), (l4, m4, g4) = got
    assert abs(l4 - l1) <= 1e-5 * l1
    assert np.abs(m4 - m1).max() <= 4096 * 2.0 ** -24 * np.abs(m1).max()
    assert np.linalg.norm(g4 - g1) <= 0.05 * np.linalg.norm(g1)
    # and a last pass of one record
    m, g = got[0][1:]
    cache.train(np.concatenate([rec, rec[:1]]), np.concatenate([tg, tg[:1]]), grad_only=True)
    m2, g2 = cache.get_gradients()
    assert np.abs(m2 - m).max() <= 0.047 * np.abs(m).max()
    assert np.linalg.norm(g2 - g) <= 0.05 * np.linalg.norm(g)


def test_a_new_cache_allocates_nothing_in_its_calls():
    """a cache's first query can be recorded into a graph, whose replays give the eager predictions, and its first
    calls leave the device's free memory as it is"""
    stream = torch.cuda.Stream()
    ctx = vk.Context(0, stream.cuda_stream)
    params = vk.default_rc_params(log2_table=14)
    n = 40000
    rec = torch.from_numpy(base.world_records(n, 27)).cuda()
    tg = torch.rand((n, 4), device="cuda")
    out, eager = (torch.zeros((n, 4), device="cuda") for _ in range(2))
    torch.cuda.synchronize()

    def query(c, o, flags=vk.DEVICE_PTRS):
        ctx.check(vk.lib().vkrt_rc_query(c.handle, rec.data_ptr(), n, o.data_ptr(), flags))

    def train(c):
        loss = ctypes.c_float()
        ctx.check(vk.lib().vkrt_rc_train(c.handle, rec.data_ptr(), tg.data_ptr(), n, vk.DEVICE_PTRS,
                                         ctypes.byref(loss)))

    warm = vk.RadianceCache(ctx, params, seed=1)  # (kernels are loaded with their first launch)
    train(warm)
    query(warm, eager)
    cache = vk.RadianceCache(ctx, params, seed=2)
    free = torch.cuda.mem_get_info()[0]
    train(cache)
    query(cache, eager)
    assert torch.cuda.mem_get_info()[0] == free
    cache = vk.RadianceCache(ctx, params, seed=3)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        query(cache, out, vk.DEVICE_PTRS | vk.ASYNC)
    for _ in range(3):
        train(cache)
        query(cache, eager)
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager) and bool(eager.any())
    del graph
    ctx.close()
