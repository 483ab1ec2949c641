"""GPU parity of small cost launches: the candidate counts around which one
pair's sets leave their own path for the staged one, sets of changing size on
one context, whose accumulators must be clean each time, and sets whose
transforms change from call to call, which the kernels read from host memory."""
import numpy as np
import pytest

import tipl_amd
from conftest import smooth_volume

pytestmark = pytest.mark.gpu


def _transforms(shape, K, seed):
    r = np.random.default_rng(seed)
    P = np.zeros((K, 12), np.float32)
    P[:, 0:3] = r.uniform(-3, 3, (K, 3))
    P[:, 3:6] = r.uniform(-0.2, 0.2, (K, 3))
    P[:, 6:9] = r.uniform(0.9, 1.1, (K, 3))
    return np.stack([tipl_amd.affine_matrix(p, shape, (1, 1, 1), shape, (1, 1, 1)) for p in P])


@pytest.mark.parametrize("kind,bins", [("mi", 256), ("mi", 64), ("corr", 256)])
def test_cost_sets_of_changing_size(ctx, oracle, kind, bins):
    shape = (14, 22, 19)
    A, B = smooth_volume(shape, 1), smooth_volume(shape, 2)
    va, vb = ctx.volume(A), ctx.volume(B)
    Ts = _transforms(shape, 64, 7)
    want = [oracle.mi_cost(A, B, t, bins) if kind == "mi" else oracle.corr_cost(A, B, t) for t in Ts]
    for K in (1, 56, 57, 3, 64, 12, 56, 1):
        got = ctx.cost_batch(va, vb, Ts[:K], kind, bins)
        # FP64 sums of the same integer counts in another order (mi), float
        # rounding of the same FP64 value (corr)
        tol = 1e-11 * np.abs(want[:K]) if kind == "mi" else np.full(K, 2.0 ** -23)
        assert (np.abs(got - want[:K]) <= tol).all(), K


def test_cost_kinds_in_turn_with_raw_counts_and_tuning(ctx, oracle):
    """Small MI and correlation sets with raw histograms, raw sums and the
    autotuner between them, which leave the accumulators full."""
    shape = (16, 20, 24)
    A, B = smooth_volume(shape, 3), smooth_volume(shape, 4)
    va, vb = ctx.volume(A), ctx.volume(B)
    Ts = _transforms(shape, 10, 9)
    mi = ctx.cost_batch(va, vb, Ts, "mi", 256)
    corr = ctx.cost_batch(va, vb, Ts, "corr")
    for _ in range(2):
        ctx.mi_hist(va, vb, Ts, 256)
        ctx.corr_sums(va, vb, Ts)
        ctx.autotune(va, vb, Ts, "corr", 256, reps=1)
        ctx.autotune(va, vb, Ts, "mi", 256, reps=1)
        assert np.array_equal(ctx.cost_batch(va, vb, Ts, "corr"), corr)
        assert np.array_equal(ctx.cost_batch(va, vb, Ts, "mi", 256), mi)
    assert abs(mi[0] - oracle.mi_cost(A, B, Ts[0])) <= 1e-11 * abs(mi[0])


@pytest.mark.parametrize("kind,bins", [("mi", 256), ("mi", 64), ("corr", 256)])
def test_largest_one_pair_sets(ctx, oracle, kind, bins):
    shape = (7, 11, 9)
    A, B = smooth_volume(shape, 5), smooth_volume(shape, 6)
    va, vb = ctx.volume(A), ctx.volume(B)
    Ts = _transforms(shape, 257, 11)
    want = np.array([oracle.mi_cost(A, B, t, bins) if kind == "mi" else oracle.corr_cost(A, B, t) for t in Ts])
    for K in (256, 257, 255):
        got = ctx.cost_batch(va, vb, Ts[:K], kind, bins)
        tol = 1e-11 * np.abs(want[:K]) if kind == "mi" else np.full(K, 2.0 ** -23)
        assert (np.abs(got - want[:K]) <= tol).all(), K


@pytest.mark.parametrize("kind,bins", [("mi", 256), ("mi", 64), ("corr", 256)])
def test_transforms_of_every_call_are_its_own(ctx, oracle, kind, bins):
    """Sets of one size, one right after the other, each with its own transforms
    (integer shifts, which the correlation crops, among them): no call may see
    the one before it."""
    shape = (12, 18, 15)
    A, B = smooth_volume(shape, 7), smooth_volume(shape, 8)
    va, vb = ctx.volume(A), ctx.volume(B)
    sets = [_transforms(shape, 3, 20 + i) for i in range(8)]
    for i, Ts in enumerate(sets):
        Ts[i % 3] = [1, 0, 0, 0, 1, 0, 0, 0, 1, i - 4, 2, -i]
    want = [[oracle.mi_cost(A, B, t, bins) if kind == "mi" else oracle.corr_cost(A, B, t) for t in Ts]
            for Ts in sets]
    got = [ctx.cost_batch(va, vb, Ts, kind, bins) for _ in range(25) for Ts in sets]
    for i, g in enumerate(got):
        w = np.array(want[i % len(sets)])
        assert (np.abs(g - w) <= (1e-11 * np.abs(w) if kind == "mi" else 2.0 ** -23)).all(), i
