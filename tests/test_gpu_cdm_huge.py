"""The CDM loop on a volume whose packed field passes 2^32 bytes."""
import numpy as np
import pytest

from conftest import smooth_volume

pytestmark = pytest.mark.gpu


def test_field_past_4_gib_equals_its_parts(ctx):
    """715 x 708 x 708 voxels are 12 * n = 2^32 + 5.9e6 bytes a field.  The
    images are empty but for one block in the first 110 planes and its copy in
    the last 110, so the loop there is the loop on 110 planes alone: two
    iterations reach 31 planes (twelve sweeps, the smoothing and a sampled cell
    each, the gradient's window), the block is 36 planes from either cut, and
    the two blocks have one largest displacement.  The second iteration gathers
    from a field that is not zero.  The first planes are equal value for value;
    in the last the coordinates are larger and round differently (2^-15 voxel),
    which may move a sampled byte by one: the bar of whole runs."""
    d, h, w = 715, 708, 708
    cut, block = 110, (38, 90, 80)
    assert 12 * d * h * w > 2 ** 32 > 12 * cut * h * w
    part = np.zeros((cut, h, w), np.uint8)
    part[36:36 + block[0], 40:40 + block[1], 60:60 + block[2]] = smooth_volume(block, 3, background=False)
    moved = np.roll(part, (-1, 1, 2), (0, 1, 2))

    def field(It, Is):
        vt, vs = ctx.volume(It), ctx.volume(Is)
        out = ctx.cdm_level_iterations(vt, vs, 2, want_field=True)
        vt.free()
        vs.free()
        return out

    want = field(part, moved)
    pair = np.zeros((2, d, h, w), np.uint8)
    for v, p in zip(pair, (part, moved)):
        v[:cut] = p
        v[-cut:] = p
    got = field(*pair)
    assert np.abs(want).max() > 0.5
    assert bool((got[:cut] == want).all())
    assert float(np.sqrt(((got[-cut:] - want) ** 2).sum(-1).mean())) <= 0.01 * np.sqrt(np.mean(want != 0))
    assert not got[cut:-cut].any()
