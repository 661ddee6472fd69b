"""The path tracer's launch shapes at the image sizes where the choice changes and workgroups end: the shape a
tracer chooses by itself gives the image, the segment count and the running mean of one launch per depth."""
import pytest

import vierkant_amd as vk
from test_gpu_media import _absorbing_room
from test_gpu_pt import _alpha_room
from test_gpu_textures import fully_textured_room
from test_pt_oracle_instanced import _glassy
from vierkant_amd import workloads as W

pytestmark = pytest.mark.gpu

# workgroups of 64 and 256; 131,072 lanes resident at once times 1, 2.5, 5 (two pixel groups from there) and 10
SIZES = [(1, 1), (63, 1), (255, 1), (257, 1), (33, 31), (362, 362), (331, 397), (572, 573), (573, 573), (809, 810),
         (811, 811), (1145, 1144), (1147, 1145)]


@pytest.fixture(scope="module")
def room():
    return W.room_scene(n_spheres=40)


def render(ctx, scene, size, spp, lit, tail, batches=2, depth=6):
    """the pixels' bytes and the last batch's segments; tail None: the shape the tracer chooses"""
    s = vk.default_settings()
    s.resolution[0], s.resolution[1] = size
    s.num_samples, s.max_trace_depth = spp, depth
    pt = vk.PathTracer(ctx, s, seed=9)
    if isinstance(scene, tuple):
        pt.set_instanced_scene(*scene)
    else:
        pt.set_scene(scene)
    if lit:
        pt.set_lights(W.room_lights())
    if tail is not None:
        pt.set_launch_mode(vk.PT_LAUNCH_FULL_GRID, tail)
    for _ in range(batches):
        pt.render(W.room_camera())
    got = pt.pixels().tobytes(), pt.stats().segments
    pt.close()
    return got


@pytest.mark.parametrize("lit", [False, True])
@pytest.mark.parametrize("size", SIZES)
def test_chosen_shape_gives_the_same_image(ctx, room, size, lit):
    got, want = (render(ctx, room, size, 2, lit, tail) for tail in (None, vk.PT_NO_TAIL))
    assert want[1] >= 2 * size[0] * size[1]
    assert got == want


@pytest.mark.parametrize("lit", [False, True])
@pytest.mark.parametrize("spp", [63, 64, 65, 129])
def test_runs_of_samples_give_the_same_image(ctx, room, spp, lit):
    """a small image's launches take 64 samples each"""
    got, want = (render(ctx, room, (47, 31), spp, lit, tail) for tail in (None, vk.PT_NO_TAIL))
    assert got == want


@pytest.fixture(scope="module")
def scenes():
    """the kernels' other variants: instances, alpha-tested materials, interior media, textures"""
    sc, mf, inst = W.room_instanced()
    flat = W.room_scene(n_spheres=40)
    absorbing = _absorbing_room(flat)
    return {"instanced": (_glassy(sc, mf), mf, inst), "instanced alpha": (_alpha_room(sc), mf, inst),
            "absorbing": absorbing, "absorbing instanced": (absorbing, *W.object_meshes(absorbing)),
            "textured": fully_textured_room(), "alpha": _alpha_room(flat)}


@pytest.mark.parametrize("lit", [False, True])
@pytest.mark.parametrize("size", [(47, 31), (331, 397), (811, 811)])
@pytest.mark.parametrize("name", ["instanced", "instanced alpha", "absorbing", "absorbing instanced", "textured",
                                  "alpha"])
def test_shapes_of_other_scenes_give_the_same_image(ctx, scenes, name, size, lit):
    """one lane from the camera on, a tail, and two pixel groups with a tail, against one launch per depth; and the
    smaller two images with a tail from depth 2"""
    want = render(ctx, scenes[name], size, 2, lit, vk.PT_NO_TAIL)
    assert want[1] > 2 * size[0] * size[1]
    for tail in (None, 2) if size[0] < 800 else (None,):
        assert render(ctx, scenes[name], size, 2, lit, tail) == want, tail
