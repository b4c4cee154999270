"""The surrogate network's two forms (all layers of 16 samples in one workgroup up to 512
wide, one launch per product above) at the edges of their tiles: batches around one
16-sample tile and one 32-sample step, layers whose padded width ends mid-step, and widths
on both sides of the rule.

Tolerances: those of the network's other oracle tests (bfloat16 operands rounded at the same
points, binary32 against binary64 sums): 2e-3 of the norm per layer, loss to 1e-5."""
import numpy as np
import pytest

import spacelab_amd as sl
from oracle import mlp as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_in,width,n_out,B", [
    (21, 256, 9, 15), (21, 256, 9, 16), (21, 256, 9, 17), (21, 256, 9, 33), (21, 256, 9, 257), (1, 16, 4, 1),
    (17, 272, 5, 40), (512, 80, 500, 31), (40, 512, 19, 48), (40, 528, 9, 30), (520, 64, 9, 20)])
def test_gradients_and_step(n_in, width, n_out, B):
    rng = np.random.default_rng(n_in + width + B)
    dims = [n_in, width, width, width, n_out]
    x = rng.standard_normal((B, n_in)).astype(np.float32)
    cls = rng.integers(0, 3, B).astype(np.int32)
    reg = rng.standard_normal((B, n_out - 3)).astype(np.float32)
    lr = 1e-3
    with sl.MLP(n_in, n_out, width, max_batch=B, seed=5) as m:
        w = m.get_params() + np.float32(0.02) * rng.standard_normal(m.n_params).astype(np.float32)
        m.set_params(w)
        y, p, e = m.forward(x)
        loss, g = m.gradients(x, cls, reg)
        loss_step = m.train_step(x, cls, reg, lr)
        w1 = m.get_params()
        loss1, _ = m.gradients(x, cls, reg)
        y1, _, _ = m.forward(x)
    assert loss_step == loss
    layers = M.unflatten(w.astype(np.float64), dims)
    lo, go = M.loss_and_grads(layers, x, cls, reg, emulate=True)
    assert loss == pytest.approx(lo, rel=1e-5)
    yo = M.forward(layers, x, emulate=True)[0][-1]
    assert np.abs(y - yo).max() <= 2e-3 * np.abs(yo).max()
    for k, (got, want) in enumerate(zip(M.unflatten(g.astype(np.float64), dims), go)):
        for a, o in zip(got, want):
            assert np.linalg.norm(a - o) <= 2e-3 * np.linalg.norm(o), k
    # Adam's first step from zero moments, and both bfloat16 copies follow the new weights
    expect = w - lr * g.astype(np.float64) / (np.abs(g.astype(np.float64)) + 1e-8)
    assert np.abs(w1 - expect).max() <= 2e-5 * lr + 2e-7 * np.abs(w).max()
    new = M.unflatten(w1.astype(np.float64), dims)
    yo1 = M.forward(new, x, emulate=True)[0][-1]
    assert np.abs(y1 - yo1).max() <= 2e-3 * np.abs(yo1).max()
    assert loss1 == pytest.approx(M.loss_and_grads(new, x, cls, reg, emulate=True)[0], rel=1e-5)


@pytest.mark.parametrize("n_in,width,n_out", [(21, 256, 9), (37, 1000, 10), (1500, 720, 9), (3, 1024, 2000)])
def test_parameters_exchanged_in_pieces(n_in, width, n_out):
    """Wide nets' parameters pass through pinned memory of 4 MB at a time, cut anywhere in a row:
    read back as set, and each where it belongs."""
    rng = np.random.default_rng(width)
    dims, B = [n_in, width, width, width, n_out], 3
    x = rng.standard_normal((B, n_in)).astype(np.float32)
    cls, reg = np.zeros(B, np.int32), rng.standard_normal((B, n_out - 3)).astype(np.float32)
    with sl.MLP(n_in, n_out, width, max_batch=B, seed=5) as m:
        w = m.get_params() + np.float32(0.02) * rng.standard_normal(m.n_params).astype(np.float32)
        m.set_params(w)
        assert np.array_equal(m.get_params(), w)
        y = m.forward(x)[0]
        _, g = m.gradients(x, cls, reg)
    layers = M.unflatten(w.astype(np.float64), dims)
    yo = M.forward(layers, x, emulate=True)[0][-1]
    assert np.abs(y - yo).max() <= 2e-3 * np.abs(yo).max()
    go = M.loss_and_grads(layers, x, cls, reg, emulate=True)[1]
    for k, (got, want) in enumerate(zip(M.unflatten(g.astype(np.float64), dims), go)):
        for a, o in zip(got, want):
            assert np.linalg.norm(a - o) <= 2e-3 * np.linalg.norm(o), k


@pytest.mark.parametrize("B", [1, 18, 19, 40])
def test_wide_outputs_read_in_pieces(B):
    """The layer form's outputs pass through the pinned buffer, here 18 rows of 608 at a time."""
    x = np.random.default_rng(B).standard_normal((B, 21)).astype(np.float32)
    with sl.MLP(21, 600, 16, max_batch=64, seed=2) as m:
        y, p, e = m.forward(x)
        for b in range(B):
            for all_rows, one in zip((y, p, e), m.forward(x[b:b + 1])):
                assert np.array_equal(all_rows[b], one[0]), b
