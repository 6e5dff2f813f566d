"""Shading windows sorted by closure class: a queue large enough to be sorted
(more entries than the shading grid has threads) against the same paths in
calls too small for it.  Path i draws from sequence i in either, so the
radiances must be equal bit for bit.  Scenes: one closure, every closure with
composites, and open ones with misses."""
import numpy as np
import pytest

from kazen_proto_amd import native, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["cornell", "materials", "closures", "terrain"])
@pytest.mark.parametrize("n", [300001, 1200007])
def test_sorted_windows_shade_the_same_paths(name, n):
    make = {"cornell": scenes.cornell_box, "materials": scenes.materials_scene, "closures": scenes.closures_scene,
            "terrain": lambda **k: scenes.terrain_scene(grid=64, n_spheres=24, sphere_lon=12, sphere_lat=6, **k)}[name]
    s = make(width=64, height=64, max_depth=6)
    rng = np.random.default_rng(n)
    rays = scenes.pinhole_rays(s.eye, s.lookat, s.up, s.fov_deg, 1200, 1001)[:n].copy()
    rays[:, 4:7] += rng.normal(scale=1e-3, size=(n, 3)).astype(np.float32)
    c = native.Context(0)
    c.load_scene(s)
    d = native.make_render_desc(s)
    big = c.integrate_rays(rays, d)
    st = c.render_stats()
    # the first paths of a smaller call are the same paths, shaded in order
    for m in (1000, 60000):
        part = c.integrate_rays(rays[:m], d)
        assert np.array_equal(part.view(np.uint32), big[:m].view(np.uint32)), m
    assert st["extension_rays"] >= n and np.isfinite(big).all() and big.max() > 0
    # passes of 2^16 paths (never sorted) give the whole image
    c.film_reset(512, 400)
    d2 = native.make_render_desc(s, spp=4, width=512, height=400)
    c.render_accumulate(d2)
    img = c.film_read(512, 400)
    c.set_pass_paths(1 << 16)
    c.film_reset(512, 400)
    c.render_accumulate(d2)
    assert np.array_equal(c.film_read(512, 400).view(np.uint32), img.view(np.uint32))
    c.close()
