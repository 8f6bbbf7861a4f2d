"""The traversal stack's LDS part: with as few entries as its wave-wide check can refuse, films and hits are those of
the default split."""
import numpy as np
import pytest

from noor_amd import scenes
from noor_amd.renderer import Renderer, hits_to_numpy, rays_from_numpy

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def reference():
    wl = scenes.terrain(grid=60, n_spheres=30, width=70, height=50, env_w=64, env_h=32)
    r = Renderer.from_workload(wl)
    g = np.random.default_rng(51)
    o = np.stack([g.uniform(-450, 450, 5000), g.uniform(20, 60, 5000), g.uniform(-450, 450, 5000)], 1)
    d = g.normal(size=(5000, 3))
    rays = rays_from_numpy(o.astype(np.float32), (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32))
    r.render(2)
    return r, rays, r.film(), hits_to_numpy(r.trace(rays)), hits_to_numpy(r.trace(rays, any_hit=True))


@pytest.mark.parametrize("entries", [1, 2, 3, 4, 7, 11, 64])
def test_split_does_not_change_results(reference, entries):
    r, rays, film, closest, any_hit = reference
    r.set_stack_lds(entries)
    try:
        np.testing.assert_array_equal(hits_to_numpy(r.trace(rays)), closest)
        np.testing.assert_array_equal(hits_to_numpy(r.trace(rays, any_hit=True)), any_hit)
        r.render(2, frame=1)
        np.testing.assert_array_equal(r.film(), film)
        r.render_wavefront(2, frame=1)
        np.testing.assert_array_equal(r.film(), film)
    finally:
        r.set_stack_lds(0)
