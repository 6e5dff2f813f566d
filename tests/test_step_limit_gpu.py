"""The traversal's step limit counts a ray's own node visits.  Over one
triangle (limit 67) a wave of a 2^25-ray launch handles about 6,500 rays; the
few of them that hit keep their leaf postponed until enough of the wave's rays
wait with one, through more than a hundred iterations of the others, which all
miss the root box.  No ray may run into the limit meanwhile, and exactly the
rays aimed at the triangle hit it, at t = 1."""
import numpy as np
import pytest

from kazen_proto_amd import native

pytestmark = pytest.mark.gpu

N = 1 << 25
SPARSE = 2048          # one ray in SPARSE is aimed at the triangle: about three of a wave's rays
TRI = np.array([[-1, -1, 0, 1, -1, 0, 0, 1, 0]], np.float32)


@pytest.fixture(scope="module")
def rays():
    r = np.zeros((N, 8), np.float32)
    r[:, 2], r[:, 6], r[:, 7] = -1.0, -1.0, np.inf     # in front of the triangle, looking away
    r[::SPARSE, 6] = 1.0
    return r


@pytest.mark.parametrize("two_level", [False, True])
@pytest.mark.parametrize("any_hit", [False, True])
def test_postponed_leaves_do_not_count_as_steps(rays, two_level, any_hit):
    c = native.Context(0)
    if two_level:
        c.instance_add(c.blas_add_soup(TRI), np.hstack([np.eye(3), np.zeros((3, 1))]))
        c.bvh_build(instances=native.INSTANCES_TWO_LEVEL)
    else:
        c.mesh_add_soup(TRI)
        c.bvh_build()
    rb = native.DeviceBuffer.from_array(c, rays)
    aimed = np.zeros(N, bool)
    aimed[::SPARSE] = True
    if any_hit:
        ob = native.DeviceBuffer(c, (N,), np.uint32)
        c.occluded(rb, ob)
        c.synchronize()                    # a step limit would be reported here
        assert np.array_equal(ob.numpy() != 0, aimed)
    else:
        ob = native.DeviceBuffer(c, (N, 4), np.float32)
        c.intersect_closest(rb, ob)
        c.synchronize()
        h = ob.numpy()
        assert np.array_equal(h[:, 1].view(np.uint32) == 0, aimed)
        assert np.all(h[aimed, 0] == 1.0) and np.all(np.isinf(h[~aimed, 0]))
    rb.free()
    ob.free()
    c.close()
