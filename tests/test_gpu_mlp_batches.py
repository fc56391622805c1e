"""Loss and gradient of the network at batch sizes around the row tile (16
rows), the batch splits (256 rows each, at most 32) and their remainders,
against the numpy oracle (oracle/mlp.py)."""
import numpy as np
import pytest

import rigidfibers_kth_amd as rf
from bench import layout
from oracle import mlp
from test_gpu_mlp import _random_blob, _sim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [2, 15, 16, 17, 256, 257, 272, 513, 8192, 8193, 9001])
def test_gradient_at_tile_and_split_edges(B):
    """FP32 products and sums of at most 9001 terms: 1e-4 of the largest entry
    of each parameter block, as for the small batches."""
    rng = np.random.default_rng(B)
    pos, ori = layout(20, 2e-2, 5)
    X = rng.normal(size=(B, 113)).astype(np.float32)
    Y = rng.normal(size=(B, 15)).astype(np.float32)
    w = _random_blob(17).astype(np.float32)
    with _sim(pos, ori) as sim:
        sim.mlp_set_weights(w)
        loss, g = sim.mlp_forward_backward(X, Y)
        again, g2 = sim.mlp_forward_backward(X, Y)
    assert loss == again and np.array_equal(g, g2)
    lo, go = mlp.backward(w.astype(np.float64), X.astype(np.float64), Y.astype(np.float64))
    assert loss == pytest.approx(lo, rel=2e-5)
    L = mlp.layout()
    for l in range(4):
        for key in ("W%d" % l, "b%d" % l):
            n = mlp.DIMS[l + 1] * (mlp.DIMS[l] if key[0] == "W" else 1)
            a, b = g[L[key]:L[key] + n], go[L[key]:L[key] + n]
            assert np.abs(a - b).max() <= 1e-4 * np.abs(b).max() + 1e-9, key
    assert not g[:L["first_param"]].any() and not g[L["out_mean"]:].any()
