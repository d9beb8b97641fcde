"""Network products at the edges of their buffered pieces of 128 k (one short
of one, one, one more, two and a remainder) and bias gradients past the 256
rows a workgroup sums at a time, against the CPU oracle with the tolerances of
the network's other tests (bf16 operands, FP32 sums against FP64)."""

import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import mlp_ref as R  # noqa: E402

from pguresvt import learned as Lr  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, n_in, h", [(1, 1, 16), (17, 127, 16), (16, 128, 32), (33, 129, 128), (255, 256, 16),
                                        (257, 257, 16), (513, 17, 128)])
def test_products_at_piece_edges(gpu, n, n_in, h):
    rng = np.random.default_rng(n + n_in)
    X = rng.standard_normal((n, n_in)).astype(np.float32)
    t = rng.standard_normal(n).astype(np.float32)
    p = Lr.init_params(n_in, h, n)
    p[n_in * h:n_in * h + h] = rng.standard_normal(h) * 0.1
    y = Lr.mlp_forward(p, X, n_in, h)
    ref, _ = R.forward(p, X.astype(np.float64), n_in, h)
    assert np.abs(y - ref).max() < 2e-3 * (np.abs(ref).max() + 1e-12)
    g, loss = Lr.mlp_gradient(p, X, t, n_in, h)
    gr, lr = R.gradient(p, X.astype(np.float64), t.astype(np.float64), n_in, h)
    assert abs(loss - lr) <= 1e-3 * abs(lr) + 1e-6
    offs = np.cumsum([0, n_in * h, h, h * h, h, h * h, h, h, 1])
    for a, b in zip(offs[:-1], offs[1:]):
        assert np.abs(g[a:b] - gr[a:b]).max() < 5e-3 * (np.abs(gr[a:b]).max() + 1e-12), (a, b)
