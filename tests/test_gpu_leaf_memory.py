"""Leaf statistics that the GPU would form, where it has no memory for them: the
call goes on with the host's, which are the same bit for bit
(PGSVT_FAULT=leaf:N fails the N-th buffer of their thread as out of memory)."""

import numpy as np
import pytest

import pgsvt_lib as G
from pguresvt import phantom

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nth", [1, 4])
def test_search_goes_on_with_host_leaves(gpu, monkeypatch, nth):
    # one host thread and short windows: 80 frames of 64 x 64 take the host far
    # longer than their decomposition the GPU, which then forms the leaves
    X = phantom.noisy_sequence(64, 80, drift=1, alpha=1.0, sigma=6.0, seed=12)[1]
    kw = dict(trajectory_length=3, n_jobs=1)
    Y0, e0 = G.denoise(X, **kw)
    monkeypatch.setenv("PGSVT_FAULT", "leaf:%d" % nth)
    Y1, e1 = G.denoise(X, **kw)
    assert np.array_equal(e1, e0) and np.array_equal(Y1, Y0)
