"""The adjoint's and the sample render's tiles at odd sizes.

With all light from the environment the image is linear in it, so the environment's gradient times the environment
equals the image gradient times the image: a sum over the adjoint's pixels against one that its tiles have no part in."""
import numpy as np
import pytest
import torch

from noor_amd import autograd as nag
from noor_amd import scenes
from noor_amd.renderer import Renderer
from noor_amd.scene import make_camera

pytestmark = pytest.mark.gpu

# Sums of at most 2.1M products of binary32 values, added to texels in binary32; one 64-pixel tile left out of the
# largest image changes the sum by about 3e-5.
TOL = 1e-5


@pytest.fixture(scope="module")
def scene():
    wl = scenes.adjoint_scene(subdiv=4, env_w=64, env_h=32)
    dev = torch.device("cuda:0")
    params = [torch.tensor(np.asarray(wl.info[k], np.float32), device=dev) for k in ("albedo", "roughness")]
    return Renderer.from_workload(wl), params, torch.tensor(wl.info["env"][..., :3].astype(np.float32), device=dev)


# 2-pixel tiles; 16-pixel tiles with remainders in both directions; a line; more 64-pixel tiles than resident waves;
# many per wave
@pytest.mark.parametrize("w,h", [(1, 1), (61, 47), (301, 199), (1, 8000), (701, 613), (2051, 1027)])
def test_every_pixel_counts_once(scene, w, h):
    r, params, env = scene
    r.update_camera(make_camera((0.0, 0.0, 0.95), (0.0, -0.1, -1.0), (0, 1, 0), np.radians(60.0), w, h))
    g = torch.rand((h, w, 3), generator=torch.Generator().manual_seed(5)).to(env.device) + 0.5
    for _ in range(2):  # the counters are back at zero after each launch
        e = env.clone().requires_grad_(True)
        image = nag.render(r, 1, *params, e)
        image.backward(g)
        want = (g.double() * image.detach().double()).sum().item()
        got = (e.grad.double() * env.double()).sum().item()
        assert want > 0.0 or w * h == 1  # (the one pixel sees an unlit wall)
        assert abs(got - want) <= TOL * want


@pytest.mark.parametrize("w,h", [(61, 47), (301, 199), (701, 613)])
def test_sample_is_the_film_of_one_sample(scene, w, h):
    r, params, env = scene
    r.update_camera(make_camera((0.0, 0.0, 0.95), (0.0, -0.1, -1.0), (0, 1, 0), np.radians(60.0), w, h))
    with torch.no_grad():
        image = nag.render(r, 1, *params, env).cpu().numpy()
    r.render_wavefront(1, frame=1)
    np.testing.assert_array_equal(image, r.film()[..., :3])
