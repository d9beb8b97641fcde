"""More noise items, distinct (frame, window maximum) pairs, than one launch
takes: the leaf statistics of a long sequence of small frames come in groups,
and its search gives what a search of its first frames alone gives."""

import ctypes as C

import numpy as np
import pytest

import pgsvt_lib as G
from pguresvt import _pguresvt as P

pytestmark = pytest.mark.gpu


def test_long_sequence_of_small_frames(gpu):
    n, nf, t = 16, 4500, 15
    rng = np.random.default_rng(2)
    X = np.asfortranarray(rng.poisson(30.0, (n, n, nf)).astype(np.float64))
    # the last frame of a window holds its maximum, so no two windows share one
    X[3, 4, :] = 200.0 + 0.01 * np.arange(nf)
    assert (nf - t) * t > 65536
    kw = dict(trajectory_length=t, patch_overlap=4, n_jobs=4)
    Y, est = G.denoise(X, **kw)
    # the first windows alone: few enough items for the host to form theirs
    f = P.load().pgsvt_denoise_range
    f.argtypes = ([C.c_void_p, C.c_int] + [C.c_uint32] * 3 + [C.POINTER(P.pgsvt_params)] + [C.c_uint32] * 2 +
                  [C.c_void_p, C.c_void_p])
    k = 32
    Yk, ek = np.zeros((n, n, k), order="F"), np.zeros((k, 4), order="F")
    p = G.params(**kw)
    P.check(f(X.ctypes.data, 3, n, n, nf, C.byref(p), 0, k, Yk.ctypes.data, ek.ctypes.data))
    assert np.array_equal(est[:k], ek) and np.array_equal(Y[:, :, :k], Yk)
