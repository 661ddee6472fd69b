"""Brute force at the sizes where its tiles (32 triangles, 32 rays a lane pair), stages of 256 triangles, workgroups
of 128 and 512 rays and triangle chunks end, and on inputs whose magnitudes its filter cannot bound: every record and
flag is the oracle's, bit for bit."""
import time

import numpy as np
import pytest
import torch

import oracle_binding as orc
from parity import assert_hits_equal
from vierkant_amd import workloads as W

pytestmark = pytest.mark.gpu


def soup(rng, n_tri, n_ray, centre=0.0, scale=1.0):
    """n_tri triangles in a cube about `centre`, and rays through it, some of them with a short or empty interval"""
    size = 2.0 * n_tri ** (-1 / 3)
    tris = rng.uniform(-1, 1, (n_tri, 1, 3)) + rng.uniform(-size, size, (n_tri, 3, 3))
    o = rng.uniform(-2, 2, (n_ray, 3))
    d = rng.uniform(-0.8, 0.8, (n_ray, 3)) - o
    rays = W.make_rays((o * scale + centre).astype(np.float32), W.glm_normalize(d.astype(np.float32)))
    rays["tmin"][::7] = 0.5 * scale
    rays["tmax"][::5] = 1.5 * scale
    rays["tmax"][::11] = 0.25 * scale
    return (tris * scale + centre).astype(np.float32).reshape(n_tri, 9), rays


def check(ctx, tris, rays, label):
    want = orc.brute_closest(tris, rays)
    assert_hits_equal(ctx.brute_closest(tris, rays), want, label)
    assert np.array_equal(ctx.brute_any(tris, rays), orc.brute_any(tris, rays)), label
    return want


@pytest.mark.parametrize("n_ray", [1, 31, 33, 127, 128, 129, 513])
@pytest.mark.parametrize("n_tri", [1, 2, 31, 32, 33, 255, 256, 257, 511, 2049])
def test_brute_at_tile_edges(ctx, n_tri, n_ray):
    rng = np.random.default_rng(n_tri * 1000 + n_ray)
    check(ctx, *soup(rng, n_tri, n_ray), f"{n_tri} triangles, {n_ray} rays")


def test_brute_with_128_rays_a_wave(ctx):
    """40,001 rays and 53 stages of 256 triangles and one more: waves of 128 rays, a chunk of two stages; the
    oracle's records for rays of the first and the last workgroups"""
    tris, rays = soup(np.random.default_rng(5), 53 * 256 + 1, 40001)
    pick = np.r_[0:600, 39000:40001]
    want = orc.brute_closest(tris, rays[pick])
    assert (want["prim"] != 0xFFFFFFFF).sum() > 300
    assert_hits_equal(ctx.brute_closest(tris, rays)[pick], want, "128 rays a wave")
    assert np.array_equal(ctx.brute_any(tris, rays)[pick], orc.brute_any(tris, rays[pick]))


@pytest.mark.parametrize("centre,scale", [(0.0, 1e-6), (0.0, 1e6), (0.0, 1e13), (0.0, 1e19), (1e4, 1.0), (1e6, 1.0),
                                          (-3e7, 10.0)])
def test_brute_over_magnitudes(ctx, centre, scale):
    """scenes from tiny to past the filter's limit, and far from the origin, where coordinates are coarse"""
    check(ctx, *soup(np.random.default_rng(9), 700, 400, centre, scale), f"{centre} {scale}")


@pytest.mark.parametrize("distance", [1e2, 1e3, 1e5, 1e8, 1e14])
def test_brute_from_far_away(ctx, distance):
    """rays whose origins lie far from the triangles, with directions from tiny to long"""
    rng = np.random.default_rng(15)
    tris, rays = soup(rng, 600, 500)
    d = rng.normal(size=(500, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    o = -distance * d + rng.uniform(-0.7, 0.7, (500, 3))
    d *= 10.0 ** rng.integers(-25, 6, (500, 1))
    for k, axis in enumerate("xyz"):
        rays["o" + axis], rays["d" + axis] = o[:, k].astype(np.float32), d[:, k].astype(np.float32)
    rays["tmin"], rays["tmax"] = 0.0, np.inf
    want = check(ctx, tris, rays, f"from {distance}")
    if distance < 1e5:
        assert (want["prim"] != 0xFFFFFFFF).sum() > 30


def test_brute_with_large_small_and_non_finite(ctx):
    """triangles of 1e-3 beside ones of 1e5, sparse NaNs, infinities and huge vertices, directions of any length, and
    rays with NaN or infinite parts or intervals: the first triangle of a chunk among them"""
    rng = np.random.default_rng(12)
    tris, rays = soup(rng, 900, 600)
    tris[100:120] *= np.float32(1e5)
    tris[200:300] = tris[200:300, :1] + (tris[200:300] - tris[200:300, :1]) * np.float32(1e-3)
    for bad in (np.nan, np.inf, -np.inf, 3e38):
        tris[rng.integers(0, 900, 6), rng.integers(0, 9, 6)] = bad
    tris[0, 0], tris[512, 2] = np.nan, np.inf
    for f in ("dx", "dy", "dz"):
        rays[f][:200] *= (10.0 ** rng.uniform(-6, 6, 200)).astype(np.float32)
    for f, bad in (("ox", np.nan), ("dy", np.inf), ("dz", 0.0), ("tmin", np.nan), ("tmax", np.nan), ("tmin", -np.inf),
                   ("oy", 3e38), ("dx", 1e30)):
        rays[f][rng.integers(0, 600, 8)] = bad
    want = check(ctx, tris, rays, "mixed")
    assert (want["prim"] != 0xFFFFFFFF).sum() > 100


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf, 1e30])
@pytest.mark.parametrize("where", ["first", "middle", "last", "ends", "tile", "all"])
def test_brute_stray_triangles(ctx, bad, where):
    """non-finite and far-off vertices where a chunk takes its origin from, in a whole tile, and everywhere; and rays with
    such parts, tmin below zero among them (an infinite direction then gives t = +-0)"""
    rng = np.random.default_rng(31)
    tris, rays = soup(rng, 512 + 40, 300)
    at = {"first": [0, 256, 512], "middle": [128, 276, 384], "last": [255, 511, 551], "ends": [0, 276, 551],
          "tile": slice(64, 96), "all": slice(None)}[where]
    tris[at, rng.integers(0, 9)] = bad
    rays["tmin"][::3] = -1.0
    for k, f in enumerate(("ox", "oy", "oz", "dx", "dy", "dz")):
        rays[f][10 + k::40] = bad
    check(ctx, tris, rays, f"{bad} {where}")


def test_brute_non_finite_parts_cost_no_more(ctx):
    """65,536 rays and the 20,480-triangle icosphere with every 256th triangle and every 32nd ray NaN take about as long
    as without (a chunk, or a wave, that gives its filter up for them takes four times as long and more)"""
    pos, idx, rays = W.icosphere_rays(65536)
    tris = W.flat_triangles(pos, idx).astype(np.float32)
    times = []
    for bad in (False, True):
        if bad:
            tris, rays = tris.copy(), rays.copy()
            tris[::256, 0] = np.nan
            rays["ox"][::32] = np.nan
        t = torch.from_numpy(tris).cuda()
        r = torch.from_numpy(rays.view(np.float32).reshape(-1, 8).copy()).cuda()
        out = torch.zeros((65536, 4), dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        best = float("inf")
        for _ in range(12):
            t0 = time.perf_counter()
            ctx.brute_closest(t, r, out=out)
            best = min(best, time.perf_counter() - t0)
        times.append(best)
    assert times[1] < 2.5 * times[0], times
