"""The film fold at pixel counts and sample counts around its tile (64 pixels,
16 samples): the same films as the batch renderer's own fold, bit for bit, and
as passes split by accumulating a few samples at a time."""
import numpy as np
import pytest

from kazen_proto_amd import native, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height,spp", [(1, 1, 1), (7, 5, 1), (13, 11, 3), (8, 8, 16), (9, 7, 17), (33, 2, 40),
                                              (65, 1, 15), (16, 12, 32)])
def test_film_fold_edges(width, height, spp):
    s = scenes.cornell_box(width=width, height=height, spp=spp, max_depth=3)
    c, owner = native.Context(0), native.Context(0)
    c.load_scene(s)
    d = native.make_render_desc(s)
    img = c.render(d)
    b = native.Batch(owner, [c])
    b.render([d])
    assert np.array_equal(b.film_read(0, width, height).view(np.uint32), img.view(np.uint32))
    c.film_reset(width, height)
    for first in range(spp):
        c.render_accumulate(native.make_render_desc(s, spp=1, spp_offset=first))
    assert np.array_equal(c.film_read(width, height).view(np.uint32), img.view(np.uint32))
    b.close()
    c.close()
    owner.close()
