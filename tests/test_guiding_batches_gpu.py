"""Training batches around the kernel's group (64 samples), chunk (16) and grid
sizes.  The gradient of a batch is the sum of its samples' gradients: with the
weights multiplied by the batch size, the mean's factor cancels to about one
float rounding, which moves a bfloat16 output gradient to its neighbour
(2^-8 relative) with probability about 2^-24 / 2^-9, so a batch and the sum of
its parts agree to about 2^-8 sqrt(2^-15) = 2e-5 in the 2-norm; 2e-4 is allowed."""
import numpy as np
import pytest

from kazen_proto_amd import native

pytestmark = pytest.mark.gpu


def _samples(n, seed):
    rng = np.random.default_rng(seed)
    unit = lambda v: v / np.linalg.norm(v, axis=1, keepdims=True)
    in6 = np.concatenate([rng.random((n, 3)), unit(rng.normal(size=(n, 3)))], 1).astype(np.float32)
    return in6, unit(rng.normal(size=(n, 3))).astype(np.float32), rng.uniform(0.5, 2.0, n).astype(np.float32)


def _grad(c, in6, dirs, w):
    return c.guiding_train_step(in6, dirs, w * np.float32(len(w)), apply=False).astype(np.float64)


@pytest.fixture(scope="module")
def ctx():
    c = native.Context(0)
    c.guiding_init(11)
    rng = np.random.default_rng(12)
    c.guiding_set_params((c.guiding_get_params() * 1.7 + rng.uniform(-0.05, 0.05, c.GUIDE_PARAMS)).astype(np.float32))
    yield c
    c.close()


@pytest.mark.parametrize("n", [2, 15, 16, 17, 63, 64, 65, 129])
def test_small_batch_is_the_sum_of_its_samples(ctx, n):
    in6, dirs, w = _samples(n, n)
    total = sum(_grad(ctx, in6[i:i + 1], dirs[i:i + 1], w[i:i + 1]) for i in range(n))
    got = _grad(ctx, in6, dirs, w)
    for a, b in ((0, 3136), (3136, 7296), (7296, 11456), (11456, 15616), (15616, 17696)):   # the layers
        assert np.linalg.norm(got[a:b] - total[a:b]) <= 2e-4 * np.linalg.norm(total[a:b])


@pytest.mark.parametrize("n,cut", [(32768, 64), (32769, 32704), (262144, 100000)])
def test_large_batch_is_the_sum_of_its_parts(ctx, n, cut):
    in6, dirs, w = _samples(n, n)
    total = _grad(ctx, in6[:cut], dirs[:cut], w[:cut]) + _grad(ctx, in6[cut:], dirs[cut:], w[cut:])
    got = _grad(ctx, in6, dirs, w)
    assert np.linalg.norm(got - total) <= 2e-4 * np.linalg.norm(total)
    assert np.array_equal(got, _grad(ctx, in6, dirs, w))   # deterministic
