"""GPU parity of the gaussian filter's four-round launches, bit for bit, at the
edges of their 64 x 32 columns: images as wide and high as a column, a voxel
less and more, past a second column, thinner than the halo along each axis; and
bandwidths whose last rounds run singly."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.asarray(a, np.float32).view(np.uint32)


@pytest.mark.parametrize("shape", [(1, 1, 1), (6, 32, 64), (5, 31, 63), (5, 33, 65), (9, 57, 121), (2, 80, 3),
                                   (40, 2, 130), (70, 30, 20)])
@pytest.mark.parametrize("bandwidth", [4, 7, 8, 16])
def test_gaussian_march_edges(ctx, oracle, shape, bandwidth):
    rng = np.random.default_rng(bandwidth * 1000 + sum(shape))
    img = (rng.standard_normal(shape) * 300).astype(np.float32)
    field = rng.standard_normal(shape + (3,)).astype(np.float32)
    assert np.array_equal(_bits(ctx.gaussian(img, bandwidth)), _bits(oracle.gaussian(img, bandwidth)))
    assert np.array_equal(_bits(ctx.gaussian(field, bandwidth)), _bits(oracle.gaussian(field, bandwidth)))
