"""BVH builds and refits at the sizes where the build's tiles, segments and workgroups end: every invariant of
vkrt_bvh_validate, and hits equal to brute force, before and after the vertices move."""
import numpy as np
import pytest

import vierkant_amd as vk
from parity import assert_hits_equal
from vierkant_amd import workloads as W

pytestmark = pytest.mark.gpu

# leaf-box segments of 64, workgroups of 256, 512 and 1024, radix tiles, and the bounds pass's 512 x 512 grid
SIZES = [1, 2, 3, 8, 9, 63, 64, 65, 129, 255, 256, 257, 511, 513, 1023, 1024, 1025, 2047, 2049, 4097, 65537, 262145]


def check_build_and_refit(ctx, n_tri, shapes, **build):
    """a soup of n_tri triangles, built at each (leaf size, width), before and after its vertices move"""
    rng = np.random.default_rng(n_tri)
    corner = rng.uniform(-1, 1, (n_tri, 1, 3))
    size = 2.0 * n_tri ** (-1 / 3)
    pos = (corner + rng.uniform(-size, size, (n_tri, 3, 3))).astype(np.float32).reshape(-1, 3)
    idx = rng.permutation(n_tri * 3).astype(np.uint32)
    pos = np.ascontiguousarray(pos[np.argsort(idx)])
    o = rng.uniform(-2, 2, (1000, 3)).astype(np.float32)
    rays = W.make_rays(o, W.glm_normalize(rng.normal(size=(1000, 3)).astype(np.float32)))
    for leaf, width in shapes:
        bvh = ctx.bvh_build(pos, idx, max_leaf_size=leaf, width=width, **build)
        info = bvh.info()
        assert info.n_tri == n_tri and info.depth <= 64
        # a record, three indices and a place in the order per triangle; a 4-wide node and its run, or a binary one,
        # its children and its run (and room for more 4-wide nodes than there came to be)
        least = n_tri * (64 + 12 + 4) + info.n_wide_nodes * (128 + 8) + (0 if info.n_wide_nodes else info.n_nodes * 80)
        if n_tri > leaf:
            assert least <= info.device_bytes <= 2 * least + 4096
        moved = pos + np.float32(0.25) * np.sin(3.0 * pos[:, ::-1]).astype(np.float32)
        for p in (pos, moved):
            if p is moved:
                bvh.refit(p)
            check = bvh.validate(p)
            assert check["ok"], check
            assert_hits_equal(ctx.trace_closest(bvh, rays), ctx.brute_closest(W.flat_triangles(p, idx), rays),
                              f"{n_tri} triangles, leaf {leaf}, width {width}, {build}")
        bvh.close()


@pytest.mark.parametrize("builder", [vk.BUILDER_LBVH, vk.BUILDER_PLOC])
@pytest.mark.parametrize("n_tri", SIZES)
def test_build_and_refit_at_tile_edges(ctx, builder, n_tri):
    check_build_and_refit(ctx, n_tri, ((0, 0), (8, 0), (1, 2)), builder=builder)


@pytest.mark.parametrize("n_tri", [900, 1025, 2049, 65537])
@pytest.mark.parametrize("radius", [1, 3, 31, 32])
def test_ploc_radii(ctx, radius, n_tri):
    """the neighbour search's tile, span and LDS places depend on the radius: one workgroup's clusters, a few tiles and
    many"""
    check_build_and_refit(ctx, n_tri, ((0, 0), (1, 2)), builder=vk.BUILDER_PLOC, ploc_radius=radius)


@pytest.mark.parametrize("builder", [vk.BUILDER_LBVH, vk.BUILDER_PLOC])
@pytest.mark.parametrize("segments", [8, 64, 128])
def test_more_wide_nodes_than_expected(ctx, builder, segments):
    """a regular grid with one triangle a leaf has two 4-wide nodes per three triangles, more than a build makes room
    for at first: the collapse is done again, and the tree is as good as any"""
    pos, idx = vk.plane(4.0, 4.0, segments, segments)
    rng = np.random.default_rng(segments)
    o = rng.uniform(-2, 2, (1000, 3)).astype(np.float32)
    o[:, 1] = 2.0
    d = W.glm_normalize(np.column_stack([rng.uniform(-.5, .5, 1000), -np.ones(1000), rng.uniform(-.5, .5, 1000)])
                        .astype(np.float32))
    rays = W.make_rays(o, d)
    bvh = ctx.bvh_build(pos, idx, builder=builder, max_leaf_size=1)
    info = bvh.info()
    assert info.n_wide_nodes > 0.6 * info.n_tri and info.n_leaves == info.n_tri
    for lift in (0.0, 0.5):
        p = pos + np.float32([0.0, lift, 0.0]) * np.sin(pos[:, :1])
        if lift:
            bvh.refit(p)
        assert bvh.validate(p)["ok"]
        assert_hits_equal(ctx.trace_closest(bvh, rays), ctx.brute_closest(W.flat_triangles(p, idx), rays), f"{lift}")
    bvh.close()
