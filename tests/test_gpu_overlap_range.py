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
