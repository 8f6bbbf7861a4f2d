"""The persistent kernels' queue claims: ray counts at the edges of a wave, of the
least and the largest chunk of a claim; the wavefront film equals the megakernel's."""
import numpy as np
import pytest

from noor_amd import scenes
from noor_amd.renderer import Renderer
from noor_amd.scene import make_camera

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def renderer():
    return Renderer.from_workload(scenes.cornell(subdiv=3, width=64, height=64, spp=1))


# (width, height, spp): 1, 31..33 (refill threshold), 47..49 (least chunk), 63..65 (wave), 255..257 (largest chunk) rays,
# and enough rays for claims that start at the largest chunk and shrink
@pytest.mark.parametrize("w,h,spp", [(1, 1, 1), (31, 1, 1), (1, 32, 1), (33, 1, 1), (47, 1, 1), (1, 48, 1), (7, 7, 1),
                                     (9, 7, 1), (4, 4, 4), (5, 13, 1), (17, 3, 5), (16, 16, 1), (257, 1, 1),
                                     (613, 509, 13)])
def test_claims_cover_the_queue(renderer, w, h, spp):
    renderer.update_camera(make_camera((0.0, 0.0, 0.95), (0.0, -0.1, -1.0), (0, 1, 0), np.radians(60.0), w, h))
    renderer.render(spp, frame=1)
    want = renderer.film()
    renderer.reset_stats()
    renderer.render_wavefront(spp, frame=1)
    got = renderer.film()
    assert np.array_equal(want, got)
    assert renderer.stats()["extension_rays"] >= w * h * spp
