"""GPU parity of the 2-D CDM kernels at the edges of their tiles, against the
oracle."""
import numpy as np
import pytest

from test_oracle_cdm2d import field2, image2

pytestmark = pytest.mark.gpu


def _bits_equal(a, b):
    return np.array_equal(np.asarray(a, np.float32).view(np.uint32),
                          np.asarray(b, np.float32).view(np.uint32))


@pytest.mark.parametrize("shape", [(1, 1), (40, 40), (41, 39), (80, 81), (12, 200), (200, 12), (90, 1)])
def test_poisson2d_tile_edges(ctx, oracle, shape):
    """Images that end on, before and after the 40 x 40 core of a tile, and
    thinner than its halo; counts below, at and past one launch's twelve."""
    nd = field2(shape, 5, 1.0, 0.0)
    for sweeps in (11, 12, 13, 24):
        got, ml = ctx.poisson2d(nd, sweeps)
        want = nd.copy()
        oracle._c2_poisson(want, oracle._d2(want), sweeps)
        assert _bits_equal(got, want)
        assert ml == oracle.max_length2(want)


@pytest.mark.parametrize("shape", [(1, 1), (41, 39), (12, 200), (90, 1)])
def test_poisson2d_signed_zeros(ctx, oracle, shape):
    """Fields of -0.0, and of -0.0 and +0.0 mixed: a neighbour past either end of
    the array is dropped, so a -0.0 there must stay one, in the first sweep too."""
    r = np.random.default_rng(3)
    for nd in (np.full(shape + (2,), -0.0, np.float32),
               np.where(r.random(shape + (2,)) < 0.5, -0.0, 0.0).astype(np.float32)):
        for sweeps in (1, 12, 13):
            got, _ = ctx.poisson2d(nd, sweeps)
            want = nd.copy()
            oracle._c2_poisson(want, oracle._d2(want), sweeps)
            assert _bits_equal(got, want), sweeps


@pytest.mark.parametrize("shape", [(1, 1), (16, 16), (17, 15), (2, 33), (35, 1)])
def test_gradient2d_tile_edges(ctx, oracle, shape):
    """Images around the 16 x 16 tile, full-range bytes."""
    r = np.random.default_rng(sum(shape))
    Js = r.integers(0, 256, shape).astype(np.uint8)
    It = np.clip(Js.astype(int) + r.integers(-60, 61, shape), 0, 255).astype(np.uint8)
    nd, c = ctx.gradient2d(Js, It, "r")
    nd_o, c_o = oracle.gradient2(Js, It, "r")
    assert _bits_equal(nd, nd_o)
    # a sum of the same terms in another order, rounded to float
    assert abs(c - c_o) <= 2.0 ** -23 * max(abs(c_o), 1e-30)


@pytest.mark.parametrize("speed", [0.3, 3.0])
@pytest.mark.parametrize("shape", [(48, 33), (31, 95)])
def test_cdm2d_update_across_tiles(ctx, oracle, shape, speed):
    """Whole runs whose field updates sample inside and across the update's
    tiles, the running and best fields rotating: the oracle's field."""
    It = image2(shape, 21)
    Is = np.roll(It, (2, -1), (0, 1))
    ok, want, n = oracle.cdm2(It, Is, speed=speed)
    rc, got, m = ctx.cdm2d(It, Is, ctx.cdm_param(speed=speed))
    assert ok and rc == 0 and n == m
    assert float(np.sqrt(((got - want) ** 2).sum(-1).mean())) <= 0.01


@pytest.mark.parametrize("iterations", [2, 3, 5])
@pytest.mark.parametrize("shape,seed", [((16, 16), 0), ((15, 17), 0), ((17, 16), 0), ((33, 31), 0), ((16, 50), 0),
                                        ((49, 15), 0), ((2, 35), 3), ((35, 2), 20), ((1, 40), 0), ((40, 1), 0)])
def test_cdm2d_first_iterations_bit_exact(ctx, oracle, shape, seed, iterations):
    """The fused field update (accumulate, smooth, next composition) on images
    around its 16 x 16 tile and narrower, and the best field taken from among the
    rotating ones: the oracle's field after the first iterations, bit for bit, for
    one modality and for two (which compose apart).  On these images every
    iteration improves, so the last but one's update is in the result; images one
    pixel wide, where no sample is inside, keep a zero field."""
    It = image2(shape, seed, sigma=1.0, background=False)
    Is = np.roll(It, (1, -1), (0, 1))
    kw = dict(min_dimension=1000, max_iterations=iterations, speed=1.2)
    for a, b in ((It, Is), ([It, It], [Is, Is])):
        ok, want, n = oracle.cdm2(a, b, **kw)
        rc, got, m = ctx.cdm2d(a, b, ctx.cdm_param(**kw))
        assert ok and rc == 0 and n == m == iterations
        assert want.any() or min(shape) == 1
        assert _bits_equal(got, want)
