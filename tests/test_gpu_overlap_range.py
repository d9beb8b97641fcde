"""The FP32 overlap-add over a wide range of values: sums are integers of a
quantum, and what is far below a window's largest value must not lose bits to
it, nor to the patches that pile up in other frames."""

import numpy as np
import pytest

import pgsvt_lib as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,patch", [(512, 4), (300, 8)])
def test_output_frame_beside_piled_up_frames(gpu, n, patch):
    # Without motion estimation every patch of the other frames lies on (0, 0):
    # 259,081 (85,849) rows on one voxel there, 4 x 4 (8 x 8) at most in the
    # frame between, which alone is put out.  All of a window is kept (plain
    # threshold 0), so that frame comes back; its dim part, 1e-8 of the rest,
    # to the accuracy of its own patches: about 30 rotations and a product of
    # 24 bits each, sqrt(30) 6e-8 = 3e-7 relative, 1e-6 with room.
    rng = np.random.default_rng(n)
    X = 1e-8 * (1 + rng.random((n, n, 3)))
    X[n // 2:, n // 2:, 1] = 0.5 + 0.5 * rng.random((n - n // 2, n - n // 2))
    X = np.asfortranarray(X / X.max())
    g = G.window_reconstruct(X, 1, 0.0, trajectory_length=3, patch_size=patch, motion_estimation=False,
                             exponential_weighting=False)
    dim = np.s_[:n // 2 - patch, :, 1]
    assert G.rel_l2(g[dim], X[dim]) < 1e-6
    assert G.rel_l2(g[:, :, 1], X[:, :, 1]) < 1e-6


def _patch_average(X, patch, gain):
    """Patches of one frame times gain(norm), averaged over each voxel (FP64)."""
    n = X.shape[0]
    P = np.lib.stride_tricks.sliding_window_view(X, (patch, patch))
    g = gain(np.sqrt((P * P).sum(axis=(2, 3))))
    out, W = np.zeros((n, n)), np.zeros((n, n))
    m = n - patch + 1
    for r in range(patch):
        for c in range(patch):
            out[r:r + m, c:c + m] += g * P[:, :, r, c]
            W[r:r + m, c:c + m] += 1
    return out / W


# One-frame windows: a patch is one column, its own leading vector, and comes
# back as d x with d = (s - lambda) / s; three roundings and an average,
# 4 * 6e-8 relative, 1e-6 with room.
ONE = dict(trajectory_length=1, motion_estimation=False, exponential_weighting=False)


@pytest.mark.parametrize("n,patch", [(96, 4), (250, 4), (96, 5), (200, 8)])
def test_sixteen_decades_in_a_frame(gpu, n, patch):
    rng = np.random.default_rng(n + patch)
    band = n // 16
    k = np.minimum(np.arange(n) // band, 15)
    X = np.asfortranarray((10.0 ** -k[:, None] * (0.5 + 0.5 * rng.random((n, n))))[:, :, None])
    X /= X.max()
    g = G.window_reconstruct(X, 0, 0.0, patch_size=patch, **ONE)[:, :, 0]
    rel = np.abs(g / X[:, :, 0] - 1)
    # a voxel at the edge shares a row of its patch with the brighter band;
    # all others are held for themselves
    inner = (np.arange(n) % band >= patch - 1) | (k == 0) | (np.arange(n) >= 16 * band)
    assert inner.sum() >= 16 and rel[inner].max() < 1e-6


def test_columns_past_the_range(gpu):
    # lambda = -1000 makes every patch 1,000 long, whatever its own length
    # (1e-6 to 1 here): 30 to 250 times the bound that follows from s_0
    rng = np.random.default_rng(8)
    n = 64
    X = np.asfortranarray((10.0 ** -(6 * rng.random((n, n)))))[:, :, None]
    X /= X.max()
    g = G.window_reconstruct(X, 0, -1000.0, **ONE)[:, :, 0]
    want = _patch_average(X[:, :, 0], 4, lambda s: (s + 1000) / s)
    assert G.rel_l2(g, want) < 1e-6


def test_rows_that_are_not_finite(gpu):
    # patches of about 1e-21: s^2 is an FP32 denormal, 1 / s^2 infinite, and
    # so is v_0: their rows are the sign's infinity, NaN where the value is 0
    rng = np.random.default_rng(9)
    n = 48
    X = 0.5 + 0.5 * rng.random((n, n))
    tiny = 3e-21 * (1 + rng.random((20, 20))) * rng.choice([-1.0, 1.0], (20, 20))
    tiny[5, 7] = tiny[11, 12] = 0.0
    X[:20, :20] = tiny
    X = np.asfortranarray((X / X.max())[:, :, None])
    g = G.window_reconstruct(X, 0, 0.0, **ONE)[:, :, 0]
    with np.errstate(invalid="ignore"):
        want = np.sign(tiny) * np.inf
    assert np.array_equal(g[:20, :20], want, equal_nan=True)
    far = np.ones((n, n), bool)
    far[:20, :20] = False
    assert np.isfinite(g[far]).all()
    assert np.abs(g[far] / X[:, :, 0][far] - 1).max() < 1e-6
