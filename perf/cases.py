"""The work that a program has this library do, as cases that can be timed and whose results can be compared.

A case is a dict of plain values; its "kind" is one of

  closest     closest hits of rays through one mesh BVH (vkrt_trace_closest)
  any         any-hit shadow rays through one mesh BVH (vkrt_trace_any)
  brute       closest hits without an acceleration structure (vkrt_intersect_brute_closest)
  batch       closest hits of many scenes in one launch (vkrt_batch_launch)
  build       a mesh BVH from scratch (vkrt_bvh_build), then a few rays through it
  refit       a mesh BVH refitted to moved vertices (vkrt_bvh_refit), then a few rays through it
  scene       closest hits through a two-level scene (vkrt_scene_trace_closest)
  path        one batch of the path tracer over the room scene (vkrt_pt_render), with or without analytic lights
  cache       one training step of the radiance cache and a query of it (vkrt_rc_train, vkrt_rc_query)

Meshes are the heightfield with icospheres of the closest-hit benchmark, at other sizes too, and the path
tracer's room. Rays, vertices and results live in device memory (torch tensors), as in a renderer that keeps
its data on the GPU. Hit records are returned as the 32-bit words they are: the library promises the same bits
for any acceleration structure and visiting order.
"""
import ctypes
import functools
import math

import numpy as np
import torch

import vierkant_amd as vk
from vierkant_amd import workloads as W

MAX_LEAF = 2            # triangles per leaf, as the closest-hit benchmark builds
TRIS_PER_SPHERE = 1280  # IcoSphere(r, 3)
EYE = (0.0, 3.0, 7.0)
MLP_SHAPES = [(64, 64)] * 5 + [(16, 64)]


@functools.lru_cache(maxsize=None)
def context():
    """the program's one context, on its own stream"""
    return vk.Context(0)


# -- cases -----------------------------------------------------------------------------------------
def listed():
    return [
        # a picking ray bundle or a handful of visibility rays against one object: the call's own latency counts
        {"name": "closest_small", "kind": "closest", "rays": 4096, "grid": 0, "spheres": 1, "bounce": False},
        # the closest-hit benchmark's step: 2048 x 2048 camera rays and as many cosine bounce rays over 1.8M
        # triangles
        {"name": "closest_frame", "kind": "closest", "rays": 4194304, "grid": 512, "spheres": 1000, "bounce": True},
        # the shadow rays of a smaller frame, an odd number of them
        {"name": "any_shadow", "kind": "any", "rays": 2073601, "grid": 512, "spheres": 1000},
        # the brute-force configuration: 65,536 rays against the 20,480-triangle jittered icosphere
        {"name": "brute_icosphere", "kind": "brute", "rays": 65536, "subdiv": 5},
        # many uneven scenes drained by one launch
        {"name": "batch_scenes", "kind": "batch", "scenes": 32, "max_tris": 200000, "max_rays": 524288},
        # one mesh of a scene being loaded or streamed in, with the default builder
        {"name": "build_small", "kind": "build", "grid": 96, "spheres": 8, "ploc": False, "leaf": 0},
        # the benchmark scene's tree: 1.8M triangles, the quality builder
        {"name": "build_scene", "kind": "build", "grid": 512, "spheres": 1000, "ploc": True, "leaf": MAX_LEAF},
        # a deforming mesh of that size, every frame
        {"name": "refit_scene", "kind": "refit", "grid": 512, "spheres": 1000, "ploc": True, "leaf": MAX_LEAF},
        # the two-level version of the benchmark scene: 1,001 instances of two meshes, camera and bounce rays
        {"name": "scene_frame", "kind": "scene", "rays": 1048576, "grid": 512, "spheres": 1000, "bounce": True},
        # one full-HD batch of the path tracer
        {"name": "path_frame", "kind": "path", "width": 1920, "height": 1080, "spp": 16, "depth": 8, "lit": False},
        # a preview at an odd size with the room's six analytic lights (shadow rays, multiple importance sampling)
        {"name": "path_lit_preview", "kind": "path", "width": 957, "height": 539, "spp": 4, "depth": 8, "lit": True},
        # the radiance cache's step: a training batch, then the queries of a frame
        {"name": "cache_step", "kind": "cache", "train": 16384, "query": 262144, "log2_table": 19},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["closest", "any", "brute", "batch", "build", "refit", "scene", "path", "cache"])
    grid = _log_int(rng, 8, 512)
    mesh = {"grid": grid, "spheres": _log_int(rng, 1, 1000)}
    if kind == "closest":
        return dict(mesh, kind=kind, rays=_log_int(rng, 64, 4194304), bounce=rng.random() < 0.5)
    if kind == "any":
        return dict(mesh, kind=kind, rays=_log_int(rng, 64, 4194304))
    if kind == "brute":
        return {"kind": kind, "rays": _log_int(rng, 256, 65536), "subdiv": rng.randint(1, 5)}
    if kind == "batch":
        return {"kind": kind, "scenes": rng.randint(3, 32), "max_tris": _log_int(rng, 2000, 200000),
                "max_rays": _log_int(rng, 32768, 524288)}
    if kind in ("build", "refit"):
        return dict(mesh, kind=kind, ploc=rng.random() < 0.5, leaf=rng.choice([0, 1, 2, 4, 8]))
    if kind == "scene":
        return dict(mesh, kind=kind, rays=_log_int(rng, 64, 1048576), bounce=rng.random() < 0.5)
    if kind == "path":
        lit = rng.random() < 0.5
        return {"kind": kind, "width": rng.randint(160, 1280), "height": rng.randint(90, 720),
                "spp": rng.randint(1, 6), "depth": rng.randint(3, 8), "lit": lit}
    return {"kind": kind, "train": _log_int(rng, 256, 65536), "query": _log_int(rng, 256, 1048576),
            "log2_table": rng.randint(14, 19)}


# -- inputs ----------------------------------------------------------------------------------------
def _heightfield(grid, seed):
    """the benchmark's displaced plane at another resolution: positions [n, 3], indices"""
    pos, idx = vk.plane(10.0, 10.0, grid, grid)
    pos[:, 1] = (0.2 * W.fbm(pos[:, 0], pos[:, 2], seed=seed)).astype(np.float32)
    return pos, idx


def _placements(n, seed):
    """centers and radii of the benchmark's icospheres: log-uniform radii, hovering over the heightfield"""
    u = np.random.default_rng(seed).uniform(size=(n, 4))
    radii = 0.01 * 10.0 ** u[:, 0]
    cx, cz = 10.0 * u[:, 1] - 5.0, 10.0 * u[:, 2] - 5.0
    cy = 0.2 * W.fbm(cx, cz, seed=seed) + u[:, 3]
    return np.stack([cx, cy, cz], axis=1), radii


def _mesh(case, seed):
    """the case's triangles as one indexed mesh; grid 0 is icospheres alone, around the origin"""
    unit, uidx = vk.icosphere(1.0, 3)
    n = case["spheres"]
    if case["grid"]:
        pos, idx = _heightfield(case["grid"], seed)
        centers, radii = _placements(n, seed)
    else:
        pos, idx = np.zeros((0, 3), np.float32), np.zeros(0, np.uint32)
        centers, radii = np.random.default_rng(seed).uniform(-0.5, 0.5, (n, 3)), np.ones(n)
    sp = (unit[None] * radii[:, None, None] + centers[:, None, :]).astype(np.float32).reshape(-1, 3)
    base = len(pos) + np.arange(n, dtype=np.uint32)[:, None] * np.uint32(len(unit))
    return np.concatenate([pos, sp]), np.concatenate([idx, (uidx[None, :] + base).reshape(-1)]).astype(np.uint32)


def _n_tri(case):
    return 2 * case["grid"] ** 2 + TRIS_PER_SPHERE * case["spheres"]


def _probe_rays(case):
    """rays that show what a build or a refit left: a quarter of its triangles' number, a frame's part at most"""
    return max(4096, min(262144, _n_tri(case) // 4))


def _device(a):
    a = np.ascontiguousarray(a)
    return torch.from_numpy(a.view(np.int32) if a.dtype == np.uint32 else a).cuda()


def _rays(o, d, tmin=0.0):
    """(n, 8) float32 rays: origin, tmin, unit direction, tmax = inf"""
    r = torch.empty((len(d), 8), device="cuda")
    r[:, :3], r[:, 3], r[:, 4:7], r[:, 7] = o, tmin, torch.nn.functional.normalize(d.float(), dim=1), float("inf")
    return r


def _pinhole(n, seed):
    """the first n rays, row by row, of a square image seen from a camera near the benchmark's"""
    side = max(1, math.isqrt(n - 1) + 1)
    eye = np.asarray(EYE) + np.random.default_rng(seed).uniform(-0.2, 0.2, 3)
    fwd = -eye / np.linalg.norm(eye)
    right = np.cross(fwd, [0.0, 1.0, 0.0])
    right /= np.linalg.norm(right)
    f, r, u = (torch.from_numpy(v).cuda() for v in (fwd, right, np.cross(right, fwd)))
    th = math.tan(math.radians(50.0) * 0.5)
    k = torch.arange(n, device="cuda")
    px = ((k % side).double() + 0.5) / side * 2.0 - 1.0
    py = 1.0 - (torch.div(k, side, rounding_mode="floor").double() + 0.5) / side * 2.0
    d = f[None] + (px * th)[:, None] * r[None] + (py * th)[:, None] * u[None]
    return _rays(torch.from_numpy(eye).cuda().float(), d)


def _surface(primary, hits, pos, idx):
    """where camera rays met the mesh: whether they did, the point moved off the surface, the facing normal"""
    prim = hits[:, 3].long()
    hit = hits[:, 3] != -1
    t = torch.where(hit, hits[:, 0].view(torch.float32), torch.zeros((), device="cuda")).double()
    v = pos[idx.view(-1, 3)[torch.where(hit, prim, 0)].long()].double()
    nrm = torch.linalg.cross(v[:, 1] - v[:, 0], v[:, 2] - v[:, 0])
    nrm = nrm / nrm.norm(dim=1, keepdim=True).clamp_min(1e-30)
    d = primary[:, 4:7].double()
    nrm = torch.where(((nrm * d).sum(1) > 0)[:, None], -nrm, nrm)
    p = primary[:, :3].double() + t[:, None] * d
    return hit, torch.where(hit[:, None], p + 1e-4 * nrm, primary[:, :3].double()), nrm


def _bounce(primary, hits, pos, idx, seed):
    """cosine-distributed rays off the surfaces that the camera rays met; a miss keeps its ray"""
    hit, o, nrm = _surface(primary, hits, pos, idx)
    g = torch.Generator(device="cuda").manual_seed(seed + 1)
    u = torch.rand((len(primary), 2), generator=g, device="cuda", dtype=torch.float64)
    r, phi = u[:, 0].sqrt(), 2.0 * math.pi * u[:, 1]
    up = torch.zeros_like(nrm)
    up[:, 0] = (nrm[:, 0].abs() <= 0.9).double()
    up[:, 1] = 1.0 - up[:, 0]
    tx = torch.nn.functional.normalize(torch.linalg.cross(up, nrm), dim=1)
    ty = torch.linalg.cross(nrm, tx)
    d = (r * phi.cos())[:, None] * tx + (r * phi.sin())[:, None] * ty + (1.0 - u[:, 0]).clamp_min(0).sqrt()[:, None] * nrm
    d = torch.where(hit[:, None], d, primary[:, 4:7].double())
    return _rays(o.float(), d, torch.where(hit, 1e-4, 0.0))


def _hits(n):
    return torch.zeros((n, 4), dtype=torch.int32, device="cuda")


def _build(case, pos, idx):
    torch.cuda.synchronize()
    return context().bvh_build(pos, idx, builder=vk.BUILDER_PLOC if case.get("ploc", True) else vk.BUILDER_LBVH,
                               max_leaf_size=case.get("leaf", MAX_LEAF))


class _DeviceRays:
    """a torch tensor as a batch item's buffer: a device address and a length"""

    def __init__(self, tensor):
        self.tensor, self.ptr = tensor, tensor.data_ptr()

    def __len__(self):
        return len(self.tensor)


def _batch(case, seed):
    # how large each scene is belongs to the case; what is in it, to the seed
    sizes = np.random.default_rng(case["scenes"])
    items, outs = [], []
    for k in range(case["scenes"]):
        n_tri = math.exp(sizes.uniform(math.log(1000), math.log(case["max_tris"])))
        n_ray = int(math.exp(sizes.uniform(math.log(16384), math.log(case["max_rays"]))))
        pos, idx = _mesh({"grid": max(1, round(math.sqrt(n_tri / 4.0))),
                          "spheres": max(1, round(n_tri / 2560.0))}, seed + k)
        lo, hi = torch.from_numpy(pos.min(0)).cuda(), torch.from_numpy(pos.max(0)).cuda()
        g = torch.Generator(device="cuda").manual_seed(seed + k)
        o = 0.5 * (lo + hi) + (torch.rand((n_ray, 3), generator=g, device="cuda") * 1.5 - 0.75) * (hi - lo)
        r = _rays(o, torch.randn((n_ray, 3), generator=g, device="cuda"))
        h = _hits(n_ray)
        bvh = _build({"ploc": False, "leaf": 0}, _device(pos), _device(idx))
        items.append((bvh, _DeviceRays(r), _DeviceRays(h)))
        outs.append(h)
    torch.cuda.synchronize()
    return {"batch": vk.Batch(context(), items), "items": items, "out": outs}


def _records(n, seed):
    """surface points as the path tracer hands them to the cache: position, roughness | view direction,
    metalness | normal, transmission | albedo"""
    rng = np.random.default_rng(seed)
    r = np.zeros((n, 16), np.float32)
    r[:, 0:3] = rng.uniform(0.0, 1.0, (n, 3))
    r[:, 3] = rng.uniform(0.05, 1.0, n)
    for k in (4, 8):
        d = rng.normal(size=(n, 3))
        r[:, k:k + 3] = d / np.linalg.norm(d, axis=1, keepdims=True)
    r[:, 7] = rng.uniform(0.0, 1.0, n) < 0.3
    r[:, 12:15] = rng.uniform(0.0, 1.0, (n, 3))
    return r


def _weights(log2_table, seed):
    """a cache part-way through a frame's training: the matrices at their usual scale, table entries of 0.1"""
    rng = np.random.default_rng(seed)
    mlp = [rng.uniform(-1.0, 1.0, s) * math.sqrt(6.0 / (s[0] + s[1])) for s in MLP_SHAPES]
    mlp[-1][3:] = 0.0
    grid = rng.random(16 * 2 ** log2_table * 2, dtype=np.float32) * np.float32(0.2) - np.float32(0.1)
    return np.concatenate([m.reshape(-1) for m in mlp]).astype(np.float32), grid


def _cache_inputs(case, seed):
    mlp, grid = _weights(case["log2_table"], seed)
    train, query = _records(case["train"], seed + 1), _records(case["query"], seed + 2)
    targets = np.zeros((case["train"], 4), np.float32)
    targets[:, :3] = np.random.default_rng(seed + 3).uniform(0.0, 2.0, (case["train"], 3))
    return mlp, grid, train, targets, query


def prepare(case, seed):
    ctx, kind = context(), case["kind"]
    s = {"case": case}
    if kind == "brute":
        g = torch.Generator(device="cuda").manual_seed(seed)
        pos, idx = W.jittered_icosphere(case["subdiv"], seed=seed)
        s["tris"] = _device(W.flat_triangles(pos, idx))
        o = torch.rand((case["rays"], 3), generator=g, device="cuda") * 6.0 - 3.0
        s["rays"] = _rays(o, torch.randn((case["rays"], 3), generator=g, device="cuda"))
        s["out"] = _hits(case["rays"])
    elif kind == "batch":
        s.update(_batch(case, seed))
    elif kind == "scene":
        pos, idx = _heightfield(case["grid"], seed)
        unit, uidx = vk.icosphere(1.0, 3)
        meshes = [(_device(pos), _device(idx)), (_device(unit), _device(uidx))]
        s["meshes"] = [_build(case, *m) for m in meshes]
        inst = [vk.instance(np.eye(3, 4), 0)]
        for k, (c, r) in enumerate(zip(*_placements(case["spheres"], seed))):
            inst.append(vk.instance(np.column_stack([np.eye(3) * r, c]), 1, custom_index=k + 1))
        s["scene"] = vk.Scene(ctx, s["meshes"], np.array(inst, dtype=vk.INSTANCE_DTYPE))
        s["rays"] = [_pinhole(case["rays"], seed)]
        s["out"] = [torch.zeros((case["rays"], 8), dtype=torch.int32, device="cuda") for _ in range(1 + case["bounce"])]
        if case["bounce"]:
            # bounce rays start where the same triangles as one mesh are met
            fpos, fidx = (_device(a) for a in _mesh(case, seed))
            flat, hits = _build({}, fpos, fidx), _hits(case["rays"])
            ctx.trace_closest(flat, s["rays"][0], out=hits)
            s["rays"].append(_bounce(s["rays"][0], hits, fpos, fidx, seed))
            torch.cuda.synchronize()
            flat.close()
    elif kind == "path":
        st = vk.default_settings()
        st.resolution[0], st.resolution[1] = case["width"], case["height"]
        st.num_samples, st.max_trace_depth = case["spp"], case["depth"]
        s["pt"] = vk.PathTracer(ctx, st, seed=seed)
        s["pt"].set_scene(W.room_scene(seed=seed))
        if case["lit"]:
            s["pt"].set_lights(W.room_lights())
        s["camera"] = W.room_camera()
        s["out"] = torch.zeros((case["height"] * case["width"], 8), dtype=torch.int32, device="cuda")
    elif kind == "cache":
        mlp, grid, train, targets, query = _cache_inputs(case, seed)
        s["cache"] = vk.RadianceCache(ctx, vk.default_rc_params(log2_table=case["log2_table"]), seed=seed)
        s["cache"].set_params(mlp, grid)
        s["train"], s["targets"], s["query"] = (_device(a) for a in (train, targets, query))
        s["out"] = torch.zeros((case["query"], 4), device="cuda")
    else:
        pos, idx = (_device(a) for a in _mesh(case, seed))
        if kind in ("build", "refit"):
            s["rays"], s["out"] = _pinhole(_probe_rays(case), seed), _hits(_probe_rays(case))
            s["pos"], s["idx"] = pos, idx
            if kind == "refit":
                s["bvh"] = _build(case, pos, idx)
                # a swell through the whole mesh
                s["pos"] = pos.clone()
                s["pos"][:, 1] += 0.1 * torch.sin(2.0 * pos[:, 0] + 0.1 * (seed % 60)) * torch.cos(1.5 * pos[:, 2])
        else:
            s["bvh"], primary = _build(case, pos, idx), _pinhole(case["rays"], seed)
            s["rays"], s["out"] = [primary], [_hits(case["rays"])]
            if kind == "any" or case["bounce"]:
                hits = _hits(case["rays"])
                torch.cuda.synchronize()
                ctx.trace_closest(s["bvh"], primary, out=hits)
                if kind == "any":
                    hit, o, _ = _surface(primary, hits, pos, idx)
                    light = torch.tensor([[0.3, 1.0, 0.2]], device="cuda").expand(len(o), 3)
                    s["rays"] = [_rays(o.float(), light, torch.where(hit, 1e-4, 0.0))]
                    s["out"] = [torch.zeros(case["rays"], dtype=torch.uint8, device="cuda")]
                else:
                    s["rays"].append(_bounce(primary, hits, pos, idx, seed))
                    s["out"].append(_hits(case["rays"]))
    torch.cuda.synchronize()
    return s


# -- passes ----------------------------------------------------------------------------------------
def run(s):
    ctx, kind = context(), s["case"]["kind"]
    if kind == "closest":
        # (a frame queues its launches and goes on; a lone small bundle is waited for)
        flags = vk.ASYNC if len(s["rays"]) > 1 else 0
        for rays, out in zip(s["rays"], s["out"]):
            ctx.trace_closest(s["bvh"], rays, out=out, flags=flags)
        return s["out"]
    if kind == "any":
        ctx.trace_any(s["bvh"], s["rays"][0], out=s["out"][0], flags=vk.ASYNC)
        return s["out"]
    if kind == "brute":
        return ctx.brute_closest(s["tris"], s["rays"], out=s["out"], flags=vk.ASYNC)
    if kind == "batch":
        s["batch"].launch(flags=vk.ASYNC)
        return s["out"]
    if kind == "build":
        bvh = _build_in_place(s)
        ctx.trace_closest(bvh, s["rays"], out=s["out"])
        info = bvh.info()
        bvh.close()
        return {"hits": s["out"], "bounds": [float(x) for x in info.bounds], "n_tri": int(info.n_tri)}
    if kind == "refit":
        s["bvh"].refit(s["pos"])
        ctx.trace_closest(s["bvh"], s["rays"], out=s["out"])
        return {"hits": s["out"], "bounds": [float(x) for x in s["bvh"].info().bounds]}
    if kind == "scene":
        for rays, out in zip(s["rays"], s["out"]):
            s["scene"].trace_closest(rays, out=out, flags=vk.ASYNC)
        return s["out"]
    if kind == "path":
        # a frame of a moving camera: accumulation restarts, the pixels stay on the GPU
        pt = s["pt"]
        pt.reset_accumulator()
        pt.render(s["camera"])
        ctx.check(vk.lib().vkrt_pt_read_pixels(pt._h, s["out"].data_ptr(), vk.DEVICE_PTRS))
        words = s["out"]
        return {"radiance": words[:, :5].view(torch.float32), "info": words[:, 5:]}
    cache, lib, loss = s["cache"], vk.lib(), ctypes.c_float()
    n = s["case"]["train"]
    ctx.check(lib.vkrt_rc_train(cache.handle, s["train"].data_ptr(), s["targets"].data_ptr(), n, vk.DEVICE_PTRS,
                                ctypes.byref(loss)))
    ctx.check(lib.vkrt_rc_query(cache.handle, s["query"].data_ptr(), s["case"]["query"], s["out"].data_ptr(),
                                vk.DEVICE_PTRS))
    grad = np.zeros(cache.n_mlp, np.float32)
    ctx.check(lib.vkrt_rc_get_gradients(cache.handle, grad.ctypes.data, None))
    return {"loss": loss.value, "mlp_gradient": grad, "prediction": s["out"][:, :3]}


def _build_in_place(s):
    c = s["case"]
    return context().bvh_build(s["pos"], s["idx"], builder=vk.BUILDER_PLOC if c["ploc"] else vk.BUILDER_LBVH,
                               max_leaf_size=c["leaf"])


# -- what a pass cannot do without -----------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "closest":
        # 32-B rays in, 16-B records out, 48-B triangle records read once
        k = 1 + case["bounce"]
        return {"bytes": 48 * case["rays"] * k + 48 * _n_tri(case), "flops": 0}
    if kind == "any":
        return {"bytes": 33 * case["rays"] + 48 * _n_tri(case), "flops": 0}
    if kind == "brute":
        n = 20 * 4 ** case["subdiv"]
        return {"bytes": 36 * n + 48 * case["rays"], "flops": 52 * n * case["rays"]}  # 52 operations a test
    if kind == "batch":
        mean = lambda lo, hi: (hi - lo) / math.log(hi / lo)  # noqa: E731  (of a log-uniform size)
        return {"bytes": case["scenes"] * (48 * mean(16384, case["max_rays"]) + 48 * mean(1000, case["max_tris"])),
                "flops": 0}
    if kind in ("build", "refit"):
        # 36 B of vertices and 12 B of indices in, a 48-B record and a 64-B node out per triangle, and the probes
        return {"bytes": 160 * _n_tri(case) + 48 * _probe_rays(case), "flops": 0}
    if kind == "scene":
        k = 1 + case["bounce"]
        return {"bytes": 64 * case["rays"] * k + 48 * (2 * case["grid"] ** 2 + TRIS_PER_SPHERE), "flops": 0}
    if kind == "path":
        # the scene's 276,504 triangles (48-B records and 36 B of normals), and 32-B pixels written once
        return {"bytes": 84 * 276504 + 32 * case["width"] * case["height"], "flops": 0}
    # 80 B a training record and 80 B a query, 512 B of table entries each (none more often than the table holds
    # it); 43,008 operations forward, three times that for a training record
    table = 64 * 2 ** case["log2_table"]
    n, q = case["train"], case["query"]
    return {"bytes": 80 * (n + q) + min(table, 512 * n) + min(table, 512 * q), "flops": 43008 * (3 * n + q)}


def tolerance(case):
    if case["kind"] == "path":
        # the same arithmetic in the same order gives the same image; a last-place change in one transcendental
        # sends a few paths another way (the CPU integrator's own one-ulp sensitivity is 0.97 % of the mean)
        return {"rel": 0.02, "max": 0.99, "differ": 0.005}
    if case["kind"] == "cache":
        # bfloat16 matrices, and table gradients summed in binary16 in no fixed order: two passes over the same
        # inputs differ by 6e-5 (one value by 6e-3 of the mean), the gradients from 64 bits by 4e-3
        return {"rel": 0.002, "max": 0.2}
    return "exact"


# -- the cache in 64 bits --------------------------------------------------------------------------
def _encode(rec, grid, log2_table):
    """hash-grid features (16 levels x 2), spherical harmonics and the material inputs in the network's order"""
    t = 1 << log2_table
    b = math.exp((math.log(2048.0) - math.log(16.0)) / 15)
    p = rec[:, :3].clamp(0.0, 1.0)
    feats = []
    for level in range(16):
        n = math.floor(16.0 * b ** level)
        x = p * n
        fl = torch.minimum(x.floor(), torch.tensor(float(n - 1), dtype=x.dtype, device=x.device))
        f, c0 = x - fl, fl.long()
        acc = torch.zeros((len(rec), 2), dtype=torch.float64, device=rec.device)
        for k in range(8):
            d = [k & 1, (k >> 1) & 1, k >> 2]
            c = [c0[:, a] + d[a] for a in range(3)]
            w = 1.0
            for a in range(3):
                w = w * (f[:, a] if d[a] else 1.0 - f[:, a])
            if (n + 1) ** 3 <= t:
                i = c[0] + (n + 1) * (c[1] + (n + 1) * c[2])
            else:
                i = (c[0] ^ (c[1] * 2654435761) ^ (c[2] * 805459861)) & (t - 1)
            acc = acc + w[:, None] * grid[level, i]
        feats.append(acc)
    x, y, z = rec[:, 4], rec[:, 5], rec[:, 6]
    xx, yy, zz, one = x * x, y * y, z * z, torch.ones_like(x)
    sh = [0.28209479177387814 * one, -0.48860251190291987 * y, 0.48860251190291987 * z, -0.48860251190291987 * x,
          1.0925484305920792 * x * y, -1.0925484305920792 * y * z, 0.94617469575755997 * zz - 0.31539156525251999,
          -1.0925484305920792 * x * z, 0.54627421529603959 * (xx - yy), 0.59004358992664352 * y * (3 * xx - yy),
          2.8906114426405538 * x * y * z, 0.45704579946446572 * y * (1 - 5 * zz),
          0.3731763325901154 * z * (5 * zz - 3), 0.45704579946446572 * x * (1 - 5 * zz),
          1.4453057213202769 * z * (xx - yy), 0.59004358992664352 * x * (xx - 3 * yy)]
    more = [rec[:, 8], rec[:, 9], rec[:, 10], rec[:, 3], rec[:, 12], rec[:, 13], rec[:, 14], rec[:, 7],
            rec[:, 11], one] + [0 * one] * 6
    cols = []
    for g in range(4):
        cols += [feats[4 * g + m] for m in range(4)]
        cols += [torch.stack(sh[4 * g:4 * g + 4], 1), torch.stack(more[4 * g:4 * g + 4], 1)]
    return torch.cat(cols, 1)


def exact(case, seed):
    """the cache's loss and matrix gradients in 64 bits. The other kinds return whole numbers (hit records as
    their bits), or images whose paths have no 64-bit counterpart; predictions follow an optimizer step whose
    first move is the sign of a gradient, which has none either"""
    if case["kind"] != "cache":
        return None
    mlp, grid, train, targets, _ = _cache_inputs(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    grid = torch.from_numpy(grid.astype(np.float64)).to(dev).view(16, -1, 2)
    w, at = [], 0
    flat = torch.from_numpy(mlp.astype(np.float64)).to(dev).requires_grad_(True)
    for shape in MLP_SHAPES:
        w.append(flat[at:at + shape[0] * shape[1]].view(shape))
        at += shape[0] * shape[1]
    h = _encode(torch.from_numpy(train.astype(np.float64)).to(dev), grid, case["log2_table"])
    for m in w[:-1]:
        h = torch.relu(h @ m.t())
    y = (h @ w[-1].t())[:, :3]
    denom = (y.mean(1, keepdim=True) ** 2 + 0.01).detach()
    loss = (((y - torch.from_numpy(targets[:, :3].astype(np.float64)).to(dev)) ** 2) / denom).sum() / case["train"]
    loss.backward()
    return {"loss": float(loss), "mlp_gradient": flat.grad.cpu(), "prediction": None}
