"""Calls whose three noise parameters are given form no leaf statistics: the
results are those of the method that still does (1 checks that a window has
enough leaves), and what was estimated can be given back."""

import numpy as np
import pytest

from pguresvt import phantom

import pgsvt_lib as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, frames", [(32, 9), (64, 6)])
def test_given_parameters_without_leaves(gpu, n, frames):
    _, X = phantom.noisy_sequence(n, frames, blobs=4, drift=1, alpha=0.8, sigma=4.0, seed=n)
    kw = dict(trajectory_length=5, noise_alpha=0.02, noise_mu=0.0, noise_sigma=0.05)
    Y1, e1 = G.denoise(X, noise_method=1, **kw)
    assert np.array_equal(e1[:, 1:], np.tile([0.02, 0.0, 0.05], (frames, 1)))
    for method in (2, 3, 4):
        Y, e = G.denoise(X, noise_method=method, **kw)
        assert np.array_equal(e, e1)
        assert np.array_equal(Y, Y1)


def test_two_given_parameters_still_estimate_the_third(gpu):
    _, X = phantom.noisy_sequence(64, 6, blobs=4, drift=1, alpha=0.8, sigma=4.0, seed=3)
    _, e = G.denoise(X, trajectory_length=5, noise_alpha=0.02, noise_mu=0.0)
    u = X[:, :, :5].astype(np.float64) / float(X[:, :, :5].max())
    sigma = G.noise_estimate(u, alpha=0.02, mu=0.0)[2]
    assert e[0, 3] == sigma


def test_too_few_leaves_are_still_refused(gpu):
    # an odd side never splits: 5 leaves, where method 1 asks for 99
    _, X = phantom.noisy_sequence(99, 6, blobs=4, drift=1, alpha=0.8, sigma=4.0, seed=99)
    with pytest.raises(Exception, match="noise method 1 needs 99 quadtree leaves"):
        G.denoise(X, noise_method=1, trajectory_length=5, noise_alpha=0.02, noise_mu=0.0, noise_sigma=0.05)
