"""A mesh whose 4-wide nodes and leaf records pass 4 GiB together (from some 41M triangles at two a leaf): the walks
then read the two from a base each. The binary tree, which no walk takes, is not kept, and every consumer's results are
brute force's or, for the path tracer, those of the same mesh as an instance."""
import numpy as np
import pytest
import torch

import vierkant_amd as vk
from vierkant_amd import workloads as W

pytestmark = pytest.mark.gpu

SIDE = 4800  # 46.1M triangles


@pytest.fixture(scope="module")
def mesh():
    """a rippled plane over [-5, 5]^2 as device tensors: positions, indices"""
    x = torch.linspace(-5, 5, SIDE + 1, device="cuda")
    z, x = torch.meshgrid(x, x, indexing="ij")
    y = 0.2 * torch.sin(3 * x) * torch.cos(2 * z) + 0.02 * torch.sin(90 * x) * torch.sin(70 * z)
    i = torch.arange(SIDE, device="cuda")
    a = (i[:, None] * (SIDE + 1) + i[None, :]).reshape(-1)
    b = a + SIDE + 1
    idx = torch.stack([a, b, a + 1, a + 1, b, b + 1], -1).to(torch.int32).reshape(-1)
    yield torch.stack([x, y, z], -1).reshape(-1, 3).contiguous(), idx.contiguous()
    torch.cuda.empty_cache()


def rays_over(n, seed):
    rng = np.random.default_rng(seed)
    o = rng.uniform((-5, 0.5, -5), (5, 2, 5), (n, 3)).astype(np.float32)
    d = W.glm_normalize(np.column_stack([rng.normal(size=n), rng.uniform(-1, 0.1, n), rng.normal(size=n)])
                        .astype(np.float32))
    return torch.from_numpy(W.make_rays(o, d).view(np.float32).reshape(n, 8).copy()).cuda()


class Device:
    """a tensor as a batch item's buffer"""

    def __init__(self, tensor):
        self.tensor, self.ptr = tensor, tensor.data_ptr()

    def __len__(self):
        return len(self.tensor)


def test_trace_batch_and_refit(ctx, mesh):
    pos, idx = mesh
    rays = rays_over(2000, 1)
    new = lambda: torch.zeros((len(rays), 4), dtype=torch.int32, device="cuda")  # noqa: E731
    torch.cuda.synchronize()
    bvh = ctx.bvh_build(pos, idx, max_leaf_size=2)
    info = bvh.info()
    assert info.n_wide_nodes * 128 + info.n_tri * 64 > 1 << 32
    assert info.device_bytes - 64 * info.n_tri - 128 * info.n_wide_nodes < 64 * info.n_nodes
    for p in (pos, pos + 0.1 * torch.sin(4.0 * pos[:, [2, 0, 1]])):
        if p is not pos:
            torch.cuda.synchronize()
            bvh.refit(p)
        tris, want, got, batched = p[idx.long()].reshape(-1, 9).contiguous(), new(), new(), new()
        occ = torch.zeros(len(rays), dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        ctx.brute_closest(tris, rays, out=want)
        ctx.trace_closest(bvh, rays, out=got)
        ctx.trace_any(bvh, rays, out=occ)
        batch = vk.Batch(ctx, [(bvh, Device(rays), Device(batched))])
        batch.launch()
        batch.close()
        hit = want[:, 3] != -1
        assert 500 < int(hit.sum()) < len(rays)
        assert torch.equal(got, want) and torch.equal(batched, want)
        assert torch.equal(occ.bool(), hit)
        del tris
    bvh.close()


def test_path_tracer(ctx, mesh):
    pos, idx = (t.cpu().numpy() for t in mesh)
    mats = np.array([vk.material((0.8, 0.7, 0.6), roughness=0.4)], dtype=vk.MATERIAL_DTYPE)
    scene = {"positions": pos, "normals": np.tile(np.float32([0, 1, 0]), (len(pos), 1)),
             "indices": idx.view(np.uint32), "tri_object": np.zeros(len(idx) // 3, np.uint32),
             "object_material": np.zeros(1, np.uint32), "materials": mats, "environment": 1.0}
    cam = vk.make_camera(eye=(0.0, 1.0, 6.0), forward=(0.0, -0.3, -1.0))
    got = []
    for two_level in (False, True):
        s = vk.default_settings()
        s.resolution[0], s.resolution[1] = 160, 90
        s.num_samples, s.max_trace_depth = 2, 4
        pt = vk.PathTracer(ctx, s, seed=3)
        if two_level:
            pt.set_instanced_scene(scene, *W.object_meshes(scene))
        else:
            pt.set_scene(scene)
        pt.set_lights(W.room_lights())
        pixels = []
        for tail in (1, vk.PT_NO_TAIL):
            pt.set_launch_mode(vk.PT_LAUNCH_FULL_GRID, tail)
            pt.reset_accumulator()
            pt.render(cam)
            pixels.append((pt.pixels().tobytes(), pt.stats().segments))
        got.append(pixels)
        pt.close()
    assert got[0][0][1] > 160 * 90 * 3
    assert got[0] == got[1]
