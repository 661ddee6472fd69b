"""The path tracer's launch shapes at the image sizes where the choice changes and workgroups end: the shape a
tracer chooses by itself gives the image, the segment count and the running mean of one launch per depth."""
import pytest

import vierkant_amd as vk
from vierkant_amd import workloads as W

pytestmark = pytest.mark.gpu

# workgroups of 64 and 256; 131,072 lanes resident at once times 1, 2.5, 5 (two pixel groups from there) and 10
SIZES = [(1, 1), (63, 1), (255, 1), (257, 1), (33, 31), (362, 362), (331, 397), (572, 573), (573, 573), (809, 810),
         (811, 811), (1145, 1144), (1147, 1145)]


@pytest.fixture(scope="module")
def room():
    return W.room_scene(n_spheres=40)


@pytest.mark.parametrize("lit", [False, True])
@pytest.mark.parametrize("size", SIZES)
def test_chosen_shape_gives_the_same_image(ctx, room, size, lit):
    got = []
    for tail in (None, vk.PT_NO_TAIL):
        s = vk.default_settings()
        s.resolution[0], s.resolution[1] = size
        s.num_samples, s.max_trace_depth = 2, 6
        pt = vk.PathTracer(ctx, s, seed=9)
        pt.set_scene(room)
        if lit:
            pt.set_lights(W.room_lights())
        if tail is not None:
            pt.set_launch_mode(vk.PT_LAUNCH_FULL_GRID, tail)
        for _ in range(2):
            pt.render(W.room_camera())
        got.append((pt.pixels().tobytes(), pt.stats().segments))
        pt.close()
    assert got[0][1] >= 2 * size[0] * size[1]
    assert got[0] == got[1]
