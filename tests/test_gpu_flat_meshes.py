"""Meshes placed by the identity (traversed with the world-space ray) beside transformed ones: structural check on the
CPU, hit queries against the oracle and films of both renderers on the GPU."""
import ctypes as C

import numpy as np
import pytest

from noor_amd import abi, scenes
from noor_amd._lib import lib
from noor_amd.renderer import Renderer, hits_to_numpy, rays_from_numpy
from noor_amd.scene import Mesh, SceneBuilder, make_camera, make_options, make_spec, material
from oracle.binding import OracleScene

TURN = np.array([[0.0, 0.0, 1.0, 0.3], [0.0, 1.0, 0.0, 0.1], [-1.0, 0.0, 0.0, -0.2]])
SHIFT = np.array([[1.0, 0.0, 0.0, 0.6], [0.0, 1.0, 0.0, 0.0], [0.0, 0.0, 1.0, 0.0]])
EYE = np.eye(4)[:3]
# (placements of the sphere, of the torus, triangles per leaf)
LAYOUTS = {
    "both_flat": ([EYE], [EYE], 2),
    "flat_and_turned": ([EYE], [TURN], 2),
    "two_identities": ([EYE, EYE], [SHIFT], 2),       # not flat: a hit has two candidate instances
    "identity_and_shift": ([EYE, SHIFT], [EYE], 2),   # the sphere is not flat, the torus is
    "leaves_of_8": ([EYE], [SHIFT], 8),               # flat leaves hold at most 4
    "none_flat": ([TURN], [SHIFT], 2),
}


def _workload(layout):
    spheres, tori, leaf = LAYOUTS[layout]
    sb = SceneBuilder()
    m = [sb.add_material(material(abi.MAT_DIFFUSE, diffuse=(0.6, 0.5, 0.4))),
         sb.add_material(material(abi.MAT_METAL, eta=scenes.CU_ETA, k=scenes.CU_K, roughness=(0.2, 0.2)))]
    sv, sf = scenes.icosphere(3)
    tp, tt, tn, tu = scenes.torus(0.8, 0.25, 24, 12)
    a = sb.add_mesh(Mesh(sv * 0.4, sf, normals=sv, material=m[0]))
    b = sb.add_mesh(Mesh(tp, tt, normals=tn, uvs=tu, material=m[1]))
    for M in spheres:
        sb.add_instance(a, M)
    for M in tori:
        sb.add_instance(b, M)
    sb.add_quad_light((-0.3, 1.5, -0.3), (0.6, 0, 0), (0, 0, 0.6), (5.0, 5.0, 5.0))
    sb.set_env(scenes.env_map(64, 32, 5))
    payload = sb.build(min_leaf=min(leaf, 2), max_leaf=leaf)
    cam = make_camera((0.0, 1.2, 2.6), (0.0, 0.0, 0.0), (0, 1, 0), np.radians(50.0), 61, 47)
    return scenes.Workload(layout, payload, cam, make_spec(payload, bounces=4), make_options(), None, 2)


@pytest.mark.parametrize("layout", LAYOUTS)
def test_wide_bvh_covers_flat_meshes(layout):
    wl = _workload(layout)
    assert lib().noor_wide_bvh_check(C.byref(wl.payload.view), None, None) == abi.OK


@pytest.mark.gpu
@pytest.mark.parametrize("layout", LAYOUTS)
def test_flat_meshes_match_oracle(layout):
    wl = _workload(layout)
    g = np.random.default_rng(41)
    o = g.normal(size=(20000, 3))
    o *= 3.0 / np.linalg.norm(o, axis=1, keepdims=True)
    d = g.uniform(-0.7, 0.7, (20000, 3)) - o
    rays = rays_from_numpy(o.astype(np.float32), d.astype(np.float32))
    for tri in (abi.TRI_WATERTIGHT, abi.TRI_WALD):
        wl.options.tri_test = tri
        r, orc = Renderer.from_workload(wl), OracleScene.from_workload(wl)
        hits = hits_to_numpy(r.trace(rays))
        assert (hits[:, 6] > 0).sum() > 5000
        np.testing.assert_array_equal(hits, hits_to_numpy(orc.trace(rays)[0]))
        np.testing.assert_array_equal(hits_to_numpy(r.trace(rays, any_hit=True))[:, 6],
                                      hits_to_numpy(orc.trace(rays, any_hit=True)[0])[:, 6])
    r.render(2)
    mega = r.film()
    np.testing.assert_array_equal(mega, orc.render(1, 2)[0])
    r.render_wavefront(2, frame=1)
    np.testing.assert_array_equal(mega, r.film())


def _empty_instance(placement):
    """A sphere placed by the identity, beside an instance of a mesh without triangles whose box is finite and in the
    way of the sphere's rays."""
    sb = SceneBuilder()
    m = sb.add_material(material(abi.MAT_DIFFUSE, diffuse=(0.6, 0.5, 0.4)))
    sv, sf = scenes.icosphere(3)
    a = sb.add_mesh(Mesh(sv * 0.4, sf, normals=sv, material=m))
    b = sb.add_mesh(Mesh(np.array([[-1.0, -1.0, -1.0], [1.0, 1.0, 1.0], [1.0, -1.0, 1.0]]), np.array([[0, 1, 2]]),
                         material=m))
    sb.add_instance(a, EYE)
    sb.add_instance(b, placement)
    sb.set_env(scenes.env_map(64, 32, 5))
    payload = sb.build()
    nodes = payload.arrays()
    leaf, only = 0x80000000, 0x80000001  # triangle leaves of the node format: the flag, and the count in the low bits
    one = np.flatnonzero(nodes["bvh_b"][:, 3] == only)
    one = [i for i in one if nodes["attr"][nodes["bvh_a"][i, 3], 0] >= len(sv)]  # the second mesh's
    assert len(one) == 1
    nodes["bvh_b"][one[0], 3] = leaf
    cam = make_camera((0.0, 1.2, 2.6), (0.0, 0.0, 0.0), (0, 1, 0), np.radians(50.0), 61, 47)
    return scenes.Workload("empty", payload, cam, make_spec(payload, bounces=4), make_options(), None, 2)


@pytest.mark.gpu
@pytest.mark.parametrize("placement", [TURN, SHIFT, EYE], ids=["turned", "shifted", "identity"])
def test_empty_instance_beside_a_flat_mesh(placement):
    wl = _empty_instance(placement)
    assert lib().noor_wide_bvh_check(C.byref(wl.payload.view), None, None) == abi.OK
    g = np.random.default_rng(42)
    o = g.normal(size=(5000, 3))
    o *= 3.0 / np.linalg.norm(o, axis=1, keepdims=True)
    rays = rays_from_numpy(o.astype(np.float32), (g.uniform(-0.4, 0.4, (5000, 3)) - o).astype(np.float32))
    r, orc = Renderer.from_workload(wl), OracleScene.from_workload(wl)
    hits = hits_to_numpy(r.trace(rays))
    assert (hits[:, 6] > 0).sum() > 1000
    np.testing.assert_array_equal(hits, hits_to_numpy(orc.trace(rays)[0]))
    np.testing.assert_array_equal(hits_to_numpy(r.trace(rays, any_hit=True))[:, 6],
                                  hits_to_numpy(orc.trace(rays, any_hit=True)[0])[:, 6])
    r.render_wavefront(2)
    np.testing.assert_array_equal(r.film(), orc.render(1, 2)[0])


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["both_flat", "flat_and_turned"])
def test_origins_with_negative_zeros(layout):
    """Origins on the sphere's vertices, their zeros written as -0, which the identity's product turns into +0: hits
    at distance zero keep the sign the oracle gives them."""
    wl = _workload(layout)
    sv, _ = scenes.icosphere(3)
    sv = (sv * 0.4).astype(np.float32)
    sv = sv[(sv == 0.0).any(1)]
    g = np.random.default_rng(43)
    o = sv[g.integers(0, len(sv), 4000)]
    o = np.where(o == 0.0, np.float32(-0.0), o)
    rays = rays_from_numpy(o, g.normal(size=(4000, 3)).astype(np.float32))
    for tri in (abi.TRI_WATERTIGHT, abi.TRI_WALD):
        wl.options.tri_test = tri
        hits = hits_to_numpy(Renderer.from_workload(wl).trace(rays))
        assert (hits[:, 6] > 0).sum() > 1000
        np.testing.assert_array_equal(hits, hits_to_numpy(OracleScene.from_workload(wl).trace(rays)[0]))


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["both_flat", "flat_and_turned", "none_flat"])
@pytest.mark.parametrize("per_wave", [1, 32, 63, 64])
def test_axis_rays_in_a_wave(layout, per_wave):
    """Rays with zero or very small direction components (the exact box test, the strict top level) as the only ones of
    their wave, as some of it and as all but one."""
    wl = _workload(layout)
    g = np.random.default_rng(45)
    n = 64 * 150
    o = g.normal(size=(n, 3))
    o *= 1.4 / np.linalg.norm(o, axis=1, keepdims=True)  # below the light: a light just behind an origin counts as hit
    d = g.uniform(-0.4, 0.4, (n, 3)) - o
    lanes = np.argsort(g.random((n // 64, 64)), axis=1).ravel() < per_wave  # that many random lanes of each wave
    small = g.choice([0.0, 2.0 ** -100, -2.0 ** -100, -2.0 ** -130], (n, 3))
    axis = g.integers(0, 3, n)
    put = lanes[:, None] & (np.arange(3)[None] == axis[:, None])
    o, d = np.where(put, g.uniform(-0.3, 0.3, (n, 3)), o), np.where(put, small, d)
    rays = rays_from_numpy(o.astype(np.float32), d.astype(np.float32))
    r, orc = Renderer.from_workload(wl), OracleScene.from_workload(wl)
    hits = hits_to_numpy(r.trace(rays))
    assert (hits[lanes, 6] > 0).sum() > lanes.sum() // 8
    np.testing.assert_array_equal(hits, hits_to_numpy(orc.trace(rays)[0]))
    np.testing.assert_array_equal(hits_to_numpy(r.trace(rays, any_hit=True))[:, 6],
                                  hits_to_numpy(orc.trace(rays, any_hit=True)[0])[:, 6])
