"""The FP32 overlap-add on large frames: strips that do not hold every row
(sides above 2,048) for small, odd and large patches, also where their sums go
by magnitude, and bins of several patch columns (sides above 8,192).  One-frame
windows: a patch is one column and comes back as d x, d = (s - lambda) / s, so
that the frame is a weighted average of patches, formed here in FP64.  Three
roundings and an average: 4 * 6e-8 relative, 1e-6 with room."""

import numpy as np
import pytest

import pgsvt_lib as G

pytestmark = pytest.mark.gpu

ONE = dict(trajectory_length=1, motion_estimation=False, exponential_weighting=False)


def _patch_average(X, patch, gain):
    n = X.shape[0]
    m = n - patch + 1
    at = [np.s_[r:r + m, c:c + m] for r in range(patch) for c in range(patch)]
    s = np.zeros((m, m))
    for q in at:
        s += X[q] ** 2
    g = gain(np.sqrt(s))
    out, W = np.zeros((n, n)), np.zeros((n, n))
    for q in at:
        out[q] += g * X[q]
        W[q] += 1
    return out / W


# lambda -1000 makes every patch 1,000 long: far past the range that follows
# from s_0, so every strip is summed by magnitude
@pytest.mark.parametrize("lam", [0.25, -1000.0])
@pytest.mark.parametrize("n,patch", [(2049, 3), (2061, 4), (2070, 8)])
def test_strips_of_cut_frames(gpu, n, patch, lam):
    rng = np.random.default_rng(n)
    X = np.asfortranarray(0.1 + 0.9 * rng.random((n, n)))
    X /= X.max()
    g = G.window_reconstruct(X[:, :, None], 0, lam, patch_size=patch, **ONE)[:, :, 0]
    want = _patch_average(X, patch, lambda s: np.maximum(s - lam, 0) / s)
    assert np.abs(g / want - 1).max() < 1e-6


def test_bins_of_two_columns(gpu):
    # step 4 covers 8,200 = 4 x 2,050 voxels a side exactly once, so the frame
    # comes back
    n = 8200
    X = np.asfortranarray(0.1 + 0.9 * np.random.default_rng(1).random((n, n), dtype=np.float32))
    X /= X.max()
    g = G.window_reconstruct(X[:, :, None], 0, 0.0, patch_overlap=4, **ONE)[:, :, 0]
    assert np.abs(g / X - 1).max() < 1e-6
