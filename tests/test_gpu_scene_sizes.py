"""Two-level scenes over mesh leaves of one to eight triangles (the first two records of a leaf are read together) and
over one to 260 instances, empty and single-leaf meshes among them: bit-exact against the oracle."""
import numpy as np
import pytest

import oracle_binding as orc
import vierkant_amd as vk
from test_gpu_scene import assert_scene_hits_equal, random_instances, scene_rays
from vierkant_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_inst", [1, 2, 5, 260])
@pytest.mark.parametrize("leaf", [1, 2, 3, 8])
def test_scene_over_leaf_sizes_and_instance_counts(ctx, leaf, n_inst):
    sphere, corner = vk.icosphere(1.0, 2), (np.eye(3, dtype=np.float32), np.arange(3, dtype=np.uint32))
    bad = (np.full((3, 3), np.nan, np.float32), np.arange(3, dtype=np.uint32))
    meshes = [sphere, vk.plane(2.0, 2.0, 5, 7), corner, bad]
    bvhs = [ctx.bvh_build(p, i, max_leaf_size=leaf) for p, i in meshes]
    tris = [W.flat_triangles(p, i) for p, i in meshes]
    inst = random_instances(n_inst, 3, seed=10 * leaf + n_inst, spread=1.0 if n_inst < 6 else 5.0)
    inst["blas"][3::7] = 3
    scene = vk.Scene(ctx, bvhs, inst)
    rays = scene_rays(1500, n_inst)
    want = orc.scene_closest(tris, inst, rays)
    assert_scene_hits_equal(scene.trace_closest(rays), want, f"leaf {leaf}, {n_inst} instances")
    assert np.array_equal(scene.trace_any(rays), (want["prim"] != 0xFFFFFFFF).astype(np.uint8))
