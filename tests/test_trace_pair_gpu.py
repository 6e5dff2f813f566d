"""The integrator's paired traversal launches (path rays and shadow rays of one
bounce together, contributions added inside the traversal) at path counts
around the wave, list and block sizes.  Path i of kp_integrate_rays draws
from sequence i whatever the call's size, so n paths must equal the first n of
a larger call bit for bit; the larger call is checked against the oracle path
by path (2e-3 relative, the tolerance of the other per-path tests)."""
import os

import numpy as np
import pytest

import oracle
from kazen_proto_amd import native, scenes

pytestmark = pytest.mark.gpu
CPU_THREADS = min(16, os.cpu_count() or 1)
N_BIG = 3001


def _scene(two_level):
    if two_level:
        return scenes.terrain_scene(grid=24, n_spheres=6, sphere_lon=12, sphere_lat=6, width=64, height=48,
                                    max_depth=5, instanced=True)
    return scenes.closures_scene(width=64, height=48, max_depth=5)


@pytest.mark.parametrize("two_level", [False, True])
@pytest.mark.parametrize("depth", [1, 5])
def test_path_counts_around_the_edges(two_level, depth):
    s = _scene(two_level)
    s.max_depth = depth
    c = native.Context(0)
    c.load_scene(s, instances=native.INSTANCES_TWO_LEVEL if two_level else native.INSTANCES_AUTO)
    rays = scenes.pinhole_rays(s.eye, s.lookat, s.up, s.fov_deg, s.width, s.height)[:N_BIG]
    d = native.make_render_desc(s)
    big = c.integrate_rays(rays, d)
    st = c.render_stats()
    od = oracle.RenderDesc()
    od.width, od.height, od.spp = s.width, s.height, 1
    od.max_depth, od.rr_depth, od.seed, od.spp_offset = s.max_depth, s.rr_depth, s.seed, 0
    od.eye[:], od.lookat[:], od.up[:] = s.eye, s.lookat, s.up
    od.tan_half_fov = s.tan_half_fov
    ref = oracle.scene_from(s).integrate_rays(rays, od, threads=CPU_THREADS)
    close = np.all(np.abs(big - ref) <= 2e-3 * np.abs(ref) + 1e-5, axis=1)
    assert close.mean() >= 0.99
    assert st["extension_rays"] >= N_BIG and 0 < st["shadow_rays"] <= st["extension_rays"]
    for n in (1, 2, 63, 64, 65, 127, 129, 255, 256, 257, 1023, 2049):
        part = c.integrate_rays(rays[:n], d)
        assert np.array_equal(part.view(np.uint32), big[:n].view(np.uint32)), n
    # a repeat gives the same bits
    assert np.array_equal(c.integrate_rays(rays, d).view(np.uint32), big.view(np.uint32))
    c.close()


COUNTS = (1, 3, 4, 5, 63, 64, 65, 1025, 4099, 8193, 32769, 65535, 65537, 131071, 131073, 327679, 327681, 655361)


def test_small_launches_split_their_rays():
    """Launches of one wave per SIMD and fewer, with rays split among lanes
    (closest hit and occlusion), at counts around each rule's limits: the host
    traversal of the same BVH gives the same bits."""
    rng = np.random.default_rng(21)
    c = native.Context(0)
    c.mesh_add_soup(scenes.microbench_triangles(seed=4, n_lon=64, n_lat=32, n_random=6000))
    c.bvh_build()
    rays = scenes.incoherent_rays(max(COUNTS), rng)
    rays[::3, 7] = rng.uniform(0.05, 1.0, rays[::3].shape[0])
    rays[5::11, 3] = -0.2
    hits, occ = c.intersect_closest_host(rays), c.occluded_host(rays)
    assert 0.2 < occ.mean() < 0.9
    for n in COUNTS:
        assert np.array_equal(c.intersect_closest(rays[:n]).view(np.uint32), hits[:n].view(np.uint32)), n
        assert np.array_equal(c.occluded(rays[:n]), occ[:n]), n
    c.close()


def test_split_occlusion_with_spilled_stacks():
    """A tree whose pending groups exceed the LDS stack: groups are handed to
    idle lanes from stacks that have spilled to memory."""
    from test_deep_bvh import deep_rays, deep_scene
    t = deep_scene()
    rays = deep_rays(3000)
    rays[1::4, 7] = 1.5
    c = native.Context(0)
    c.mesh_add_soup(t)
    c.bvh_build()
    for n in (64, 127, 2000, rays.shape[0]):
        assert np.array_equal(c.occluded(rays[:n]), c.occluded_host(rays[:n])), n
        assert np.array_equal(c.intersect_closest(rays[:n]).view(np.uint32),
                              c.intersect_closest_host(rays[:n]).view(np.uint32)), n
    c.close()


@pytest.mark.parametrize("leaf_size", [1, 2, 3, 4])
@pytest.mark.parametrize("width", [2, 5, 8])
def test_leaf_runs(leaf_size, width):
    """A leaf set is tested as the run of triangles from its first to its last
    hit slot: every leaf size with narrow nodes (empty slots) and wide ones,
    against brute force; rays from far away (boxes widened the most) and rays
    with negative starts included."""
    rng = np.random.default_rng(leaf_size * 10 + width)
    tris = scenes.small_test_scene(seed=width, n_random=900)
    rays = scenes.incoherent_rays(3000, rng)
    rays[::4, 0:3] *= 30.0
    rays[::4, 4:7] = -rays[::4, 0:3]
    rays[1::5, 3] = -0.5
    rays[2::5, 7] = 0.6
    c = native.Context(0)
    c.mesh_add_soup(tris)
    c.bvh_build(leaf_size=leaf_size, node_width=width)
    ref = oracle.closest_bruteforce(tris, rays)
    assert np.array_equal(c.intersect_closest(rays).view(np.uint32), ref.view(np.uint32))
    assert np.array_equal(c.occluded(rays) != 0, ref[:, 1].view(np.uint32) != 0xFFFFFFFF)
    c.close()
