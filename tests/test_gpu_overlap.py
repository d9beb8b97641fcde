"""The FP32 overlap-add of strips (patches up to 4 x 4) where it can go wrong:
frame sides around its strip widths and the cut at 2,048 rows, steps that
leave whole columns of positions empty, trajectories that all lie on one
position, contributions beyond its fixed-point range.  Windows against the
CPU oracle; the tolerance is the suite's for FP32 frames (1e-5 relative L2:
rows of 24-bit products, of which the overlap-add averages up to 16)."""

import numpy as np
import pytest

import oracle_lib as O
import pgsvt_lib as G
from pguresvt import phantom

pytestmark = pytest.mark.gpu
FRAME_TOL = 1e-5


def _pair(X, t, lam, **kw):
    okw = {k: int(v) if isinstance(v, bool) else v for k, v in kw.items()}
    return G.window_reconstruct(X, t, lam, **kw), O.window_reconstruct(X, t, lam, motion_filter=-1, **okw)


@pytest.mark.parametrize("n,patch,step,traj", [(5, 4, 1, 3), (15, 4, 1, 3), (16, 2, 2, 3), (17, 3, 3, 5), (33, 4, 4, 7),
                                               (127, 4, 1, 3), (129, 3, 2, 3), (257, 4, 3, 3)])
def test_strip_edges(gpu, n, patch, step, traj):
    _, X = phantom.noisy_sequence(n, traj, drift=1, alpha=1.0, sigma=6.0, seed=n)
    g, o = _pair(X, traj // 2, 1.5, patch_size=patch, patch_overlap=step, trajectory_length=traj)
    assert G.rel_l2(g, o) < FRAME_TOL


def test_rows_cut(gpu):
    # 2,049 rows: a strip of 2,048 and one of a single row
    rng = np.random.default_rng(3)
    X = np.asfortranarray(rng.random((2049, 2049, 3), dtype=np.float32))
    g, o = _pair(X, 1, 1.0, patch_size=2, patch_overlap=2, trajectory_length=3, motion_window=3)
    assert G.rel_l2(g, o) < FRAME_TOL


@pytest.mark.parametrize("n", [16, 64, 80])
def test_all_patches_on_one_position(gpu, n):
    # motion off leaves every patch of the other frames at (0, 0): 5,929 rows
    # on one voxel at n = 80, past the 2^11 that need no headroom
    _, X = phantom.noisy_sequence(n, 9, drift=0, alpha=0.5, sigma=5.0, seed=2)
    g, o = _pair(X, 4, 3.0, trajectory_length=9, motion_estimation=False)
    assert G.rel_l2(g, o) < FRAME_TOL


def test_negative_frames(gpu):
    rng = np.random.default_rng(5)
    X = np.asfortranarray((rng.normal(-300.0, 40.0, (48, 48, 5))).astype(np.float32))
    X[0, 0, 0] = 1.0  # the window's maximum: the normalised values reach -400
    # every rank kept whole gives the window back, in the frame that all
    # positions of the grid cover (the oracle takes no negative values)
    g = G.window_reconstruct(X, 2, 0.0, trajectory_length=5, exponential_weighting=False)
    assert G.rel_l2(g[:, :, 2], X[:, :, 2].astype(np.float64)) < FRAME_TOL


def test_rows_out_of_range_stay_local(gpu):
    # values of 1e-20 of the maximum: their squared singular values are FP32
    # denormals, 1 / s^2 overflows and the rows there are not finite; voxels
    # that no patch of that region covers are as ever
    rng = np.random.default_rng(6)
    X = rng.random((64, 64, 5)) + 0.5
    X[:24, :24, :] = 1e-20 * (1 + rng.random((24, 24, 5)))
    X = np.asfortranarray(X)
    g, o = _pair(X, 2, 0.0, trajectory_length=5, exponential_weighting=False)
    far = np.ones((64, 64), bool)
    far[:24 + 4 + 7, :24 + 4 + 7] = False  # patch and search reach
    assert np.isfinite(g[far]).all()
    assert G.rel_l2(g[far], o[far]) < FRAME_TOL


def test_repeated_windows_are_bit_identical(gpu):
    _, X = phantom.noisy_sequence(64, 15, drift=2, alpha=1.0, sigma=8.0, seed=9)
    a = G.window_reconstruct(X, 7, 1.0)
    r = [G.window_risk(X, 7, (0.01, 0.0, 0.03), [0.3, 1.0, 40.0]) for _ in range(2)]
    assert np.array_equal(a, G.window_reconstruct(X, 7, 1.0))
    assert np.array_equal(r[0], r[1])
