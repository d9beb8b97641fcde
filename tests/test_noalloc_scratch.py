"""Shapes that the entry point without allocation takes (no device needed):
every shape whose stated size is within the limit of 64 MiB fits the array,
and the first one above it is refused with its size."""

import ctypes as C

import pytest

import pgsvt_lib as G
from pguresvt import _pguresvt as P

LIMIT = 64 << 20


def _scratch(n, **kw):
    f = P.load().pgsvt_noalloc_scratch
    f.argtypes = [C.c_uint32] * 3 + [C.POINTER(P.pgsvt_params), C.POINTER(C.c_uint64), C.POINTER(C.c_uint64)]
    stated, held = C.c_uint64(), C.c_uint64()
    rc = f(n, n, 64, C.byref(G.params(**kw)), C.byref(stated), C.byref(held))
    return rc, stated.value, P.load().pgsvt_last_error().decode()


def _largest(kw):
    lo, hi = kw["patch_size"], 1400
    while lo < hi:
        mid = (lo + hi + 1) // 2
        if _scratch(mid, **kw)[1] <= LIMIT:
            lo = mid
        else:
            hi = mid - 1
    assert lo < 1400
    return lo


@pytest.mark.parametrize("patch", [2, 3, 4, 5, 6, 7, 8, 16])
@pytest.mark.parametrize("traj", [1, 3, 15])
def test_stated_limit_is_the_limit(patch, traj):
    for step in (1, 2):
        for optimize in (True, False):
            for median in (-1, 3):
                kw = dict(patch_size=patch, trajectory_length=traj, patch_overlap=step, optimize_pgure=optimize,
                          motion_filter=median)
                top = _largest(kw)
                for n in range(max(patch, top - 6), top + 1):
                    rc, stated, msg = _scratch(n, **kw)
                    assert rc == 0 and stated <= LIMIT, (n, kw, msg)
                rc, stated, msg = _scratch(top + 1, **kw)
                assert rc == -1 and stated > LIMIT and "bytes of device scratch" in msg, (top + 1, kw, msg)


@pytest.mark.parametrize("n,kw", [(477, dict(optimize_pgure=False)), (514, dict(optimize_pgure=False)),
                                  (331, dict()), (499, dict(optimize_pgure=False, motion_filter=3)),
                                  (544, dict(optimize_pgure=False, patch_size=3))])
def test_one_frame_windows(n, kw):
    rc, stated, msg = _scratch(n, trajectory_length=1, **kw)
    assert rc == 0 and stated <= LIMIT, msg


@pytest.mark.gpu
def test_largest_one_frame_windows_on_the_device(gpu):
    # the same frames as the entry point that allocates, in the layout that
    # takes most of the array
    import numpy as np

    from test_zz_no_alloc import _run

    X = np.random.default_rng(3).poisson(40.0, (514, 514, 2))
    kw = dict(trajectory_length=1, optimize_pgure=False, lambda1=0.5)
    Yn, en = _run("noalloc", X, **kw)
    Yd, ed = _run("device", X, **kw)
    assert np.array_equal(Yn, Yd) and np.array_equal(en, ed) and np.abs(Yn).max() > 0
