"""Hit queries where the ray set-up's range checks decide: directions scaled to both sides of the bounds of the fast
reciprocal and single components far smaller or larger than the others, bit for bit against the oracle."""
import numpy as np
import pytest

from noor_amd import abi, scenes
from noor_amd.renderer import Renderer, hits_to_numpy, rays_from_numpy
from oracle.binding import OracleScene

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pair():
    wl = scenes.cornell(subdiv=4, width=16, height=16)
    return Renderer.from_workload(wl), OracleScene.from_workload(wl)


def _rays(seed, n=6000):
    g = np.random.default_rng(seed)
    o = g.uniform(-0.95, 0.95, (n, 3))
    d = g.normal(size=(n, 3))
    return o.astype(np.float32), (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)


@pytest.mark.parametrize("any_hit", [False, True])
@pytest.mark.parametrize("axis,exponent", [(None, 0), (None, -62), (None, -59), (None, 59), (None, 62), (1, -58), (0, 30),
                                           (2, 61)])
def test_scaled_directions_bit_exact(pair, axis, exponent, any_hit):
    r, orc = pair
    o, d = _rays(31 if axis is None else 32 + axis)
    s = np.float32(2.0 ** exponent)
    if axis is None:
        d = d * s
    else:
        d[:, axis] *= s
    rays = rays_from_numpy(o, d)
    g, h = hits_to_numpy(r.trace(rays, any_hit=any_hit)), hits_to_numpy(orc.trace(rays, any_hit=any_hit)[0])
    if any_hit:
        np.testing.assert_array_equal(g[:, 6], h[:, 6])
    else:
        np.testing.assert_array_equal(g, h)


@pytest.mark.parametrize("exponent", [-129, -131, -135])
def test_overflowing_reciprocals_enter_boxes(pair, exponent):
    """Directions whose reciprocals overflow reach every box in front of them at an infinite distance: the boxes are
    entered as the reference's comparison does, and the hits, themselves at infinity, are those of the oracle."""
    r, orc = pair
    o, d = _rays(33)
    rays = rays_from_numpy(o, d * np.float32(2.0 ** exponent))
    g, h = hits_to_numpy(r.trace(rays)), hits_to_numpy(orc.trace(rays)[0])
    assert (h[:, 6] > 0).sum() > 1000
    np.testing.assert_array_equal(g, h)
    assert (hits_to_numpy(r.trace(rays, any_hit=True))[h[:, 6] > 0, 6] > 0).all()
