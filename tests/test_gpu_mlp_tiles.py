"""The training kernels at the edges of their tiles (16 rows per wave tile,
32 per weight-gradient operand, chunks of several operands): loss and
gradient against the CPU oracle with the same BF16 rounding points.  The GPU
accumulates in FP32 where the oracle uses FP64; an intermediate on the other
side of a BF16 boundary moves by 2^-8 of itself.  Each parameter block's
gradient is a sum over the rows of products of such intermediates, of which
the flips touch a small share: 2e-2 of its norm, and the loss (a sum of
squares of unflipped FP32 outputs) 1e-4."""
import numpy as np
import pytest

import mlp_oracle as mo
from batsrus_amd.core import Mlp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 15, 16, 17, 32, 33, 1023, 8193, 20000])
def test_loss_and_gradient_at_tile_edges(rows):
    print(f"case mlp gradient rows={rows}", flush=True)
    rng = np.random.default_rng(rows)
    w = (mo.init_params(seed=4) + rng.normal(0, 0.02, 27464)).astype(np.float32)
    X = rng.normal(0, 1, (rows, 16)).astype(np.float32)
    T = rng.normal(0, 1, (rows, 8)).astype(np.float32)
    with Mlp(w) as m:
        # a larger minibatch first: its operands must not reach this one's
        m.loss_grad(np.ones((rows + 40, 16)), np.ones((rows + 40, 8)))
        loss, g = m.loss_grad(X, T)
    lo, go = mo.loss_and_grad(w, X, T, rounding=True)
    assert abs(loss - lo) <= 1e-4 * lo
    o = 0
    for name, shp in mo.param_shapes():
        n = int(np.prod(shp))
        a, b = g[o:o + n].astype(np.float64), go[o:o + n]
        o += n
        rel = np.linalg.norm(a - b) / np.linalg.norm(b)
        print(f"  {name}: rel L2 {rel:.2e}")
        assert rel < 2e-2, name


@pytest.mark.parametrize("batch", [100, 1000, 3000])
def test_ragged_minibatch_training_is_deterministic(batch):
    """Minibatches that are no multiple of a tile, weighted targets off the
    device dataset: two runs give the same bits and lower the loss."""
    print(f"case mlp training batch={batch}", flush=True)
    rng = np.random.default_rng(batch)
    X = rng.uniform(-1, 1, (6011, 16)).astype(np.float32)
    T = np.tanh(X[:, :8] - X[:, 8:]).astype(np.float32)
    out = []
    for _ in range(2):
        with Mlp(mo.init_params(seed=3)) as m:
            m.set_data(X, T)
            _, e0 = m.train(0, batch=batch, hold=0.1, seed=2)
            _, e1 = m.train(4, batch=batch, lr=2e-3, hold=0.1, seed=2,
                            jump_weight=True)
            out.append((m.params()[0], e0[0], e1[0]))
    assert np.array_equal(out[0][0], out[1][0])
    assert out[0][2] < out[0][1]
