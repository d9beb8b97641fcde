"""FP64 gathers of trajectories that pile up: tiles with more patch rows than
their LDS holds form each contribution where it is summed.  Bounds as for the
FP64 path elsewhere: 1e-12 relative L2 for a window, 1e-10 relative for its
risk."""

import ctypes as C

import numpy as np
import pytest

import oracle_lib as O
import pgsvt_lib as G
from pguresvt import _pguresvt as P
from test_gpu_parity import _bowl_sequence

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("expw,lam", [(True, 0.5), (False, 0.05)])
def test_tiles_beyond_their_rows(gpu, expw, lam):
    X = _bowl_sequence(nf=16)
    kw = dict(patch_size=4, patch_overlap=1, trajectory_length=15, motion_window=7)
    L = P.load()
    L.pgsvt_set_precision.argtypes = [C.c_int]
    assert L.pgsvt_set_precision(64) == 0
    try:
        v = G.window_reconstruct(X, 8, lam, exponential_weighting=expw, **kw)
        lams, noise = [lam / 3, lam, 3 * lam], [0.02, 0.03, 0.04]
        r = G.window_risk(X, 8, noise, lams, exponential_weighting=expw, **kw)
    finally:
        assert L.pgsvt_set_precision(32) == 0
    ref = O.window_reconstruct(X, 8, lam, exponential_weighting=int(expw), motion_filter=-1, **kw)
    assert G.rel_l2(v, ref) < 1e-12
    rr = O.window_risk(X, 8, noise, lams, exponential_weighting=int(expw), motion_filter=-1, **kw)
    assert np.max(np.abs(r - rr) / np.abs(rr)) < 1e-10
