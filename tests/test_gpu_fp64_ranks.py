"""FP64 evaluations (pgsvt_set_precision(64)) of patches that keep many ranks:
a plain threshold far below most singular values, and exponential weighting
at a large lambda, whose weight falls off fast.  Bounds as for the FP64 path
elsewhere: 1e-12 relative L2 for a window (sums of 16 to 64 FP64 terms a
voxel), 1e-10 relative for its risk (differences of such sums)."""

import ctypes as C

import numpy as np
import pytest

import oracle_lib as O
import pgsvt_lib as G
from pguresvt import _pguresvt as P
from pguresvt import phantom

pytestmark = pytest.mark.gpu


@pytest.fixture
def fp64():
    L = P.load()
    L.pgsvt_set_precision.argtypes = [C.c_int]
    assert L.pgsvt_set_precision(64) == 0
    yield
    assert L.pgsvt_set_precision(32) == 0


@pytest.mark.parametrize("bs,step,traj", [(2, 1, 3), (3, 1, 9), (4, 1, 15), (4, 2, 5), (6, 2, 7), (8, 2, 15)])
@pytest.mark.parametrize("expw,lam", [(False, 0.02), (True, 500.0)])
def test_many_kept_ranks(gpu, fp64, bs, step, traj, expw, lam):
    _, X = phantom.noisy_sequence(40, 16, blobs=6, drift=1, alpha=2.0, mu=5.0, sigma=10.0, seed=4)
    kw = dict(patch_size=bs, patch_overlap=step, trajectory_length=traj)
    v = G.window_reconstruct(X, 8, lam, exponential_weighting=expw, **kw)
    ref = O.window_reconstruct(X, 8, lam, exponential_weighting=int(expw), motion_filter=-1, **kw)
    assert G.rel_l2(v, ref) < 1e-12
    lams = [0.25 * lam, lam, 4 * lam]
    noise = [0.02, 0.05, 0.03]
    r = G.window_risk(X, 8, noise, lams, exponential_weighting=expw, **kw)
    rr = O.window_risk(X, 8, noise, lams, exponential_weighting=int(expw), motion_filter=-1, **kw)
    assert np.max(np.abs(r - rr) / np.abs(rr)) < 1e-10
