"""The megakernel's tiles: images at the edges of every tile size, the film equal to the wavefront
renderer's, which has no tiles."""
import numpy as np
import pytest

from noor_amd import scenes
from noor_amd.renderer import Renderer
from noor_amd.scene import make_camera

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def renderer():
    return Renderer.from_workload(scenes.cornell(subdiv=3, width=64, height=64, spp=1))


# one pixel; lines; images of 2- to 64-pixel tiles with remainders in both directions; more tiles than resident waves
@pytest.mark.parametrize("w,h,spp", [(1, 1, 1), (1, 37, 2), (129, 1, 1), (91, 89, 2), (127, 129, 1), (181, 183, 1),
                                     (255, 257, 1), (363, 361, 1), (513, 511, 1), (1021, 769, 1)])
def test_tiles_cover_the_image(renderer, w, h, spp):
    renderer.update_camera(make_camera((0.0, 0.0, 0.95), (0.0, -0.1, -1.0), (0, 1, 0), np.radians(60.0), w, h))
    renderer.render_wavefront(spp, frame=1)
    want = renderer.film()
    for _ in range(3):  # the tile counters are back at zero after each launch
        renderer.render(spp, frame=1)
        np.testing.assert_array_equal(renderer.film(), want)


def test_groups_that_run_out_take_from_the_others(renderer):
    """An image whose rows cost very different times (sky above, the box's inside below), with many tiles per block and
    a remainder in every direction, several times in a row."""
    renderer.update_camera(make_camera((0.0, 0.9, 3.0), (0.0, 1.2, -1.0), (0, 1, 0), np.radians(80.0), 2051, 1027))
    renderer.render_wavefront(1, frame=1)
    want = renderer.film()
    for _ in range(3):
        renderer.render(1, frame=1)
        np.testing.assert_array_equal(renderer.film(), want)
