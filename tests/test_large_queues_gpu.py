"""Queues long enough to reach what small images do not: waves that finish more
shadow rays than their list of unoccluded ones holds and draw chunks from the
work counter, shading windows sorted in one pass and in the several passes of a
batch, and path depths up to the last per-bounce counters.  Path i draws from
sequence i however the paths are split over passes, so a pass of 2^16 paths (at
most 64 rays a wave, fewer entries than the shading grid has threads) must give
the same bits."""
import os

import numpy as np
import pytest

import oracle
from kazen_proto_amd import native, scenes

pytestmark = pytest.mark.gpu
CPU_THREADS = min(16, os.cpu_count() or 1)
SMALL_PASS = 1 << 16


@pytest.mark.parametrize("two_level", [False, True])
@pytest.mark.parametrize("depth", [1, 4])
def test_many_shadow_rays_a_wave(two_level, depth):
    """1.8 M paths over a small instanced terrain in one pass against passes of
    2^16: at depth 1 every shadow ray belongs to the first vertices, and there
    are more than 256 for each wave of an occlusion grid."""
    s = scenes.terrain_scene(grid=24, n_spheres=6, sphere_lon=12, sphere_lat=6, width=64, height=48,
                             max_depth=depth, instanced=True)
    c = native.Context(0)
    c.load_scene(s, instances=native.INSTANCES_TWO_LEVEL if two_level else native.INSTANCES_BAKE)
    assert c.stats()["two_level"] == int(two_level)
    # from above, so that nearly every path meets the terrain and sees a light
    rays = scenes.pinhole_rays((0.1, 9.0, 0.2), (0.0, 0.0, 0.0), (0.0, 0.0, 1.0), 50.0, 1500, 1200)
    d = native.make_render_desc(s)
    one = c.integrate_rays(rays, d)
    st = c.render_stats()
    assert st["passes"] == 1
    if depth == 1:
        assert st["shadow_rays"] > c.stats()["grid_occluded"] * 4 * 256
    c.set_pass_paths(SMALL_PASS)
    ref = c.integrate_rays(rays, d)
    st2 = c.render_stats()
    assert st2["passes"] == -(-rays.shape[0] // SMALL_PASS)
    assert np.array_equal(one.view(np.uint32), ref.view(np.uint32))
    assert (st["extension_rays"], st["shadow_rays"]) == (st2["extension_rays"], st2["shadow_rays"])
    c.close()


def _mixed(name):
    if name == "terrain":
        return scenes.terrain_scene(grid=64, n_spheres=24, sphere_lon=12, sphere_lat=6, width=256, height=256,
                                    spp=36, max_depth=5)
    make = scenes.materials_scene if name == "materials" else scenes.closures_scene
    return make(width=256, height=256, spp=24, max_depth=5)


@pytest.mark.parametrize("name", ["materials", "closures", "terrain"])
def test_sorted_shading_in_one_pass_and_in_a_batch(name):
    """A mixed-closure image whose second bounce has more entries than any
    shading grid has threads (8 blocks of 256 a CU at most), so that its
    windows are sorted, against passes of 2^16 paths, which are shaded in
    order; and the same scene twice in a batch of 2^20-path passes, with and
    without the pass graph."""
    s = _mixed(name)
    c = native.Context(0)
    c.load_scene(s)
    cus = c.stats()["device_cus"]
    n = s.width * s.height * s.spp
    d1 = native.make_render_desc(s)
    d1.max_depth = 1
    c.render(d1)
    assert c.render_stats()["extension_rays"] - n > cus * 8 * 256      # entries of the second bounce
    d = native.make_render_desc(s)
    img = c.render(d)
    st = c.render_stats()
    assert st["passes"] == 1
    c.set_pass_paths(SMALL_PASS)
    assert np.array_equal(c.render(d).view(np.uint32), img.view(np.uint32))
    st2 = c.render_stats()
    assert st2["paths_per_pass"] == SMALL_PASS
    assert (st["extension_rays"], st["shadow_rays"]) == (st2["extension_rays"], st2["shadow_rays"])
    owner = native.Context(0)
    b = native.Batch(owner, [c, c])
    for graph in (1, 0):
        b.set_tuning(pass_paths=1 << 20, use_graph=graph)
        b.render([d, d])
        assert b.stats()["passes"] == -(-2 * n // (1 << 20))
        for i in range(2):
            assert np.array_equal(b.film_read(i, s.width, s.height).view(np.uint32), img.view(np.uint32))
    b.close()
    owner.close()
    c.close()


@pytest.mark.parametrize("depth", [63, 64])
def test_depths_up_to_the_last_counters(depth):
    """A closed room of one albedo without Russian roulette: every path has
    depth + 1 segments, in renders, ray calls and batches, and paths agree with
    the oracle's (2e-3 relative, as in the other per-path tests)."""
    s = scenes.furnace_box(albedo=0.9, width=20, height=15, spp=2, max_depth=depth, rr_depth=1000)
    c, owner = native.Context(0), native.Context(0)
    c.load_scene(s)
    d = native.make_render_desc(s)
    n = s.width * s.height * s.spp
    img = c.render(d)
    st = c.render_stats()
    assert st["extension_rays"] == n * (depth + 1)
    assert 0 < st["shadow_rays"] <= n * depth
    b = native.Batch(owner, [c])
    for _ in range(3):                                   # replays of the pass graph clear the same counters
        b.render([d])
        assert b.stats()["extension_rays"] == st["extension_rays"]
        assert b.stats()["shadow_rays"] == st["shadow_rays"]
        assert np.array_equal(b.film_read(0, s.width, s.height).view(np.uint32), img.view(np.uint32))
    rays = scenes.pinhole_rays(s.eye, s.lookat, s.up, s.fov_deg, s.width, s.height)
    got = c.integrate_rays(rays, d)
    assert c.render_stats()["extension_rays"] == rays.shape[0] * (depth + 1)
    od = oracle.RenderDesc()
    od.width, od.height, od.spp = s.width, s.height, 1
    od.max_depth, od.rr_depth, od.seed, od.spp_offset = depth, s.rr_depth, s.seed, 0
    od.eye[:], od.lookat[:], od.up[:] = s.eye, s.lookat, s.up
    od.tan_half_fov = s.tan_half_fov
    ref = oracle.scene_from(s).integrate_rays(rays, od, threads=CPU_THREADS)
    close = np.all(np.abs(got - ref) <= 2e-3 * np.abs(ref) + 1e-5, axis=1)
    assert close.mean() >= 0.99
    b.close()
    owner.close()
    c.close()
