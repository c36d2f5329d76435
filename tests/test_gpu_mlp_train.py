"""The two-launch training step at the row counts where it can go wrong: around
a block's 16 rows, a matrix step's 32, a chunk's 256, and the 64 chunks past
which the weight gradients go through partial sums in memory.  Same bar as
test_gpu_learned.py: the float64 oracle that rounds to bf16 where the kernels
do, 1e-2 relative per parameter block (a bf16 rounding that falls the other
way moves a term by 2^-8 of itself), 1e-3 for the loss.
"""
import numpy as np
import pytest

from oracle import mlp as M

pytestmark = pytest.mark.gpu

BLOCKS = {"W1": (M.W1, M.B1), "b1": (M.B1, M.W2), "W2": (M.W2, M.B2), "b2": (M.B2, M.W3),
          "W3": (M.W3, M.B3), "b3": (M.B3, M.N_PARAMS)}


def rel(a, b):
    return np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-30)


@pytest.mark.parametrize("rows", [1, 15, 16, 17, 31, 32, 33, 255, 256, 257, 4099, 16384, 16385, 20011])
def test_loss_and_gradient(gpu_mod, rows):
    rng = np.random.default_rng(rows)
    params = M.random_params(rng).astype(np.float32)
    X = rng.normal(size=(rows, 32)).astype(np.float32)
    Y = rng.normal(size=(rows, 3)).astype(np.float32)
    with gpu_mod.Gpu(0) as g:
        loss, grad = g.mlp_loss_grad(params, X, Y, 0.5)
        again = g.mlp_loss_grad(params, X, Y, 0.5)
    want_loss, want = M.loss_grad(params.astype(np.float64), X, Y, 0.5, bf16_round=True)
    assert loss == pytest.approx(want_loss, rel=1e-3)
    for name, (a, b) in BLOCKS.items():
        assert rel(grad[a:b], want[a:b]) < 1e-2, name
    assert again[0] == loss and np.array_equal(again[1], grad)  # no dependence on scheduling


@pytest.mark.parametrize("batch", [32, 288, 16416])
def test_fit_steps_down(gpu_mod, batch):
    # one chunk, a partial second chunk, and 65 chunks (partial sums in memory)
    rng = np.random.default_rng(batch)
    rows = 3 * batch + 77 if batch > 1000 else 2000
    X = rng.normal(size=(rows, 32)).astype(np.float32)
    Y = (M.forward(M.random_params(rng), X, bf16_round=False)[0] * 0.02).astype(np.float32)
    with gpu_mod.Gpu(0) as g:
        t = g.trainer(rows)
        t.add(X, Y)
        tl, vl = t.fit(epochs=30, batch=batch, lr=3e-3, lr_final=1e-3, val_fraction=0.1, seed=2)
        tl2, vl2 = t.fit(epochs=30, batch=batch, lr=3e-3, lr_final=1e-3, val_fraction=0.1, seed=2)
    assert np.isfinite(tl).all() and tl[-1] < 0.7 * tl[0] and vl[-1] < vl[0]
    assert np.array_equal(tl, tl2) and np.array_equal(vl, vl2)
