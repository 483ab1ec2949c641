"""Upload statistics at the sizes where their launch can go wrong: fewer voxels
than a dword, a remainder of a dword, one workgroup and the next, extremes at
either end of the array."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 1, 1), (1, 1, 3), (2, 3, 5), (8, 32, 32), (8, 32, 33), (31, 33, 35)])
@pytest.mark.parametrize("dtype", [np.uint8, np.int16, np.float32])
def test_upload_statistics(ctx, shape, dtype):
    r = np.random.default_rng(shape[2])
    if dtype == np.float32:
        v = r.normal(0, 100, shape).astype(dtype)
    else:
        v = r.integers(0 if dtype == np.uint8 else -500, 256, shape).astype(dtype)
    if v.size > 1:
        v.flat[0], v.flat[-1] = v.min() - (dtype != np.uint8), v.max()
    vol = ctx.volume(v)
    if dtype == np.uint8:
        want = v
    else:
        lo, hi = np.float32(v.min()), np.float32(v.max())
        want = np.zeros(shape, np.uint8)
        if hi > lo:
            coef = np.float32(255.99) / np.float32(hi - lo)
            want = ((v.astype(np.float32) - lo) * coef).astype(np.uint8)
    assert np.array_equal(vol.read(), want)
    w = want.astype(np.int64)
    assert vol.stats()[:2] == (int(w.sum()), int((w * w).sum()))
    assert np.array_equal(vol.stats()[2], np.bincount(want.ravel(), minlength=256))
