"""The noise estimator's leaf statistics on the GPU round as the host's: its
sums keep the reference's even and odd chains in index order, so means and
variances are equal bit for bit, on blocks where every sum is rounding alone
(saturated and constant regions decide splits there) as on noise."""

import numpy as np
import pytest

import pgsvt_lib as G

pytestmark = pytest.mark.gpu


def _frame(kind, n):
    rng = np.random.default_rng(n)
    f = rng.random((n, n))
    if kind == "clipped":
        f = np.clip(f * 3 - 1, 0.0, 0.7)
    elif kind == "constant":
        f = np.full((n, n), 0.3)
        f[: n // 2, : n // 2] = 0.1
    elif kind == "counts":
        f = np.floor(f * 7) / 7
    elif kind == "one pixel":
        f = np.zeros((n, n))
        f[n // 3, n // 5] = 1.0
    return f


# sides: one wave a leaf (16), its edge with the workgroup's (17, 32), the
# register cache's edge (64, 65), 1,024 threads (128, 99 never split)
@pytest.mark.parametrize("kind", ["noise", "clipped", "constant", "counts", "one pixel"])
@pytest.mark.parametrize("n", [16, 17, 32, 64, 65, 99, 128, 256])
def test_leaves_equal_the_hosts(gpu, kind, n):
    mh, vh = G.frame_leaves(_frame(kind, n), False)
    mg, vg = G.frame_leaves(_frame(kind, n), True)
    assert len(mh) == len(mg) > 0
    assert np.array_equal(mg, mh, equal_nan=True)
    assert np.array_equal(vg, vh, equal_nan=True)
