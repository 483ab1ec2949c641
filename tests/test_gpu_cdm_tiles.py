"""GPU parity of the CDM kernels at the edges of their tiles and of the size
ranges their launches choose between, against the oracle."""
import numpy as np
import pytest

from conftest import smooth_volume

pytestmark = pytest.mark.gpu


def _field(shape, seed, scale=2.0, zero_frac=0.2):
    from scipy.ndimage import gaussian_filter
    r = np.random.default_rng(seed)
    d = gaussian_filter(r.standard_normal(shape + (3,)), (2, 2, 2, 0)).astype(np.float32) * scale
    d[r.random(shape) < zero_frac] = 0.0
    return d


def _bits_equal(a, b):
    return np.array_equal(np.asarray(a, np.float32).view(np.uint32),
                          np.asarray(b, np.float32).view(np.uint32))


@pytest.mark.parametrize("shape", [(1, 1, 1), (4, 4, 16), (5, 5, 17), (3, 3, 15), (9, 4, 33),
                                   (2, 11, 31), (6, 7, 2), (13, 12, 66)])
def test_gradient_tile_edges(ctx, oracle, shape):
    """Shapes that end on, before and after a 16 x 4 x 4 tile, rows that start
    at every alignment, full-range bytes: bit for bit the oracle's."""
    r = np.random.default_rng(sum(shape))
    Js = r.integers(0, 256, shape).astype(np.uint8)
    It = np.clip(Js.astype(int) + r.integers(-60, 61, shape), 0, 255).astype(np.uint8)
    nd, c = ctx.gradient(Js, It, "r")
    nd_o, c_o = oracle.gradient(Js, It, "r")
    assert _bits_equal(nd, nd_o)
    # the cost is a sum of at most n terms in another order, rounded to float
    assert abs(c - c_o) <= 2.0 ** -23 * max(abs(c_o), 1e-30)


def test_cdm_odd_levels_two_modalities(ctx, oracle):
    """A pyramid whose second modality's half-size images start at an odd
    multiple of two bytes."""
    shape = (33, 37, 41)
    A = [smooth_volume(shape, s) for s in (1, 2)]
    B = [smooth_volume(shape, s) for s in (3, 4)]
    ok, want, _ = oracle.cdm(A, B)
    rc, got, _ = ctx.cdm([ctx.volume(v) for v in A], [ctx.volume(v) for v in B])
    assert ok and rc == 0
    assert float(np.sqrt(((got - want) ** 2).sum(-1).mean())) <= 0.01


@pytest.mark.parametrize("shape", [(1, 1, 1), (8, 8, 8), (9, 7, 17), (1, 3, 40), (40, 2, 1), (16, 16, 16),
                                   (1, 1, 4096), (4096, 1, 1), (1, 1, 4097), (1030, 2, 2), (17, 16, 16),
                                   (16, 24, 11), (33, 20, 25)])
def test_poisson_four_sweep_tiles(ctx, oracle, shape):
    """Volumes of up to 4096 voxels, which take every sweep in one launch, and
    larger ones around the 8 x 8 x 8 tile of the four-sweep launch, thinner
    than its halo, and with rows shorter than it: 4, 8 and 12 sweeps, and
    remainders after four-sweep launches."""
    nd = _field(shape, 21, 1.0, 0.0)
    for sweeps in (4, 12, 5, 6, 8, 11):
        out, ml = ctx.poisson(nd, sweeps)
        want = oracle.poisson(nd, sweeps)
        assert _bits_equal(out, want), sweeps
        assert ml == oracle.max_length(want)


@pytest.mark.parametrize("shape", [(64, 64, 64), (64, 64, 65), (3, 300, 301), (300, 3, 301), (301, 300, 3),
                                   (70, 57, 113), (90, 48, 112), (1, 1, 2700000)])
def test_poisson_marched_tiles(ctx, oracle, shape):
    """The largest volume on 8 x 8 x 8 tiles and larger ones that march z:
    thinner than the halo along each axis, and with rows and planes ending on
    and inside the 56 x 24 core of a column.  13 sweeps end in a single one.
    The last: rows so long that the marched kernel's offsets would overflow."""
    nd = np.random.default_rng(5).standard_normal(shape + (3,)).astype(np.float32)
    for sweeps in (12, 13):
        out, ml = ctx.poisson(nd, sweeps)
        want = oracle.poisson(nd, sweeps)
        assert _bits_equal(out, want)
        assert ml == oracle.max_length(want)


@pytest.mark.parametrize("shape", [(16, 16, 16), (17, 19, 16), (3, 5, 300), (64, 64, 65), (3, 300, 301), (1, 1, 5000)])
def test_poisson_signed_zeros(ctx, oracle, shape):
    """Fields of -0.0, and of -0.0 and +0.0 mixed: a neighbour past either end of
    the array is dropped, so a -0.0 there must stay one, in the first sweep too,
    in the launch that takes every sweep, the tiled and the marched one."""
    r = np.random.default_rng(3)
    for nd in (np.full(shape + (3,), -0.0, np.float32),
               np.where(r.random(shape + (3,)) < 0.5, -0.0, 0.0).astype(np.float32)):
        for sweeps in (4, 12, 13):
            out, _ = ctx.poisson(nd, sweeps)
            assert _bits_equal(out, oracle.poisson(nd, sweeps)), sweeps


@pytest.mark.parametrize("speed", [0.3, 4.0])
@pytest.mark.parametrize("shape", [(21, 30, 27), (61, 67, 71), (130, 2, 1100), (1, 33, 9), (9, 1, 33), (40, 9, 1)])
def test_level_iterations_by_size(ctx, oracle, shape, speed):
    """The loop's planar gradient fields and its fused field update, on each
    side of the sizes where their kernels change, with steps inside a voxel
    and across several: the oracle's step functions in the loop's order."""
    from test_gpu_cdm import _pair, oracle_level_iterations
    It, Is = _pair(shape, 31)
    want = oracle_level_iterations(oracle, It, Is, 4, speed=speed)
    p = ctx.cdm_param(speed=speed)
    got = ctx.cdm_level_iterations(ctx.volume(It), ctx.volume(Is), 4, p, want_field=True)
    assert _bits_equal(got, want)
