"""Motion searches in tiles: trajectories equal the oracle's at frame sizes
around the tile's 64 block rows and its columns, for each kind of search (a
tile of either halo, unrolled and rolled steps, the wide window's frames)."""

import numpy as np
import pytest

from pguresvt import phantom

import oracle_lib as O
import pgsvt_lib as G

pytestmark = pytest.mark.gpu


def _clip(n, frames):
    return phantom.noisy_sequence(n, frames, blobs=5, drift=2, alpha=0.5, sigma=3.0, seed=n)[1]


# block rows a side: 61 and 64 (one tile), 65 (two of 33), 129 (three of 43);
# sides 2 .. 5 unroll, 6 .. 8 and 16 do not; windows 3, 7 (narrow tile), 9, 15
# (wide tile), 17, 31 (frames)
@pytest.mark.parametrize("n, bs, mw", [(64, 4, 7), (67, 4, 7), (68, 4, 15), (132, 4, 3), (17, 2, 9), (40, 3, 7),
                                       (69, 5, 15), (70, 6, 7), (71, 7, 9), (72, 8, 7), (72, 8, 15), (80, 16, 7),
                                       (47, 16, 15), (40, 4, 17), (50, 8, 31), (8, 8, 7), (9, 4, 15)])
def test_trajectories_equal_the_oracles(gpu, n, bs, mw):
    X = _clip(n, 7)
    kw = dict(patch_size=bs, motion_window=mw, trajectory_length=5 if bs > 2 else 3)
    for t in (0, 3, 6):
        assert np.array_equal(G.window_trajectories(X, t, **kw), O.window_trajectories(X, t, **kw)), t
