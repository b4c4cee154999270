"""Several nets through shared launches against the same nets one by one: the sums are the
same, so every comparison is of bits.  Nets laid out alike share launches, up to 16 of them;
nets of different widths or largest batch, in the layer form, or the same net twice go one by
one."""
import numpy as np
import pytest

from conftest import bits_equal

import spacelab_amd as sl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("widths,n_in,n_out,B,max_batch", [
    ([256] * 4, 21, 9, 256, [256] * 4), ([256], 21, 9, 33, [40]), ([64] * 17, 21, 9, 17, [17] * 17), ([48] * 16, 40, 40, 1, [3] * 16),
    ([256, 256, 80], 21, 9, 40, [64] * 3), ([64] * 2, 21, 9, 40, [64, 80]), ([528] * 2, 21, 9, 40, [40] * 2)])
def test_members_together_and_alone(widths, n_in, n_out, B, max_batch):
    rng = np.random.default_rng(len(widths) + B)
    rows = 3 * B
    x = rng.standard_normal((rows, n_in)).astype(np.float32)
    cls = rng.integers(0, 3, rows).astype(np.int32)
    reg = rng.standard_normal((rows, n_out - 3)).astype(np.float32)
    make = lambda: [sl.MLP(n_in, n_out, w, b, seed=k) for k, (w, b) in enumerate(zip(widths, max_batch))]
    a, b = make(), make()
    a[0].train_step(x[:B], cls[:B], reg[:B], 1e-3)      # the nets need not be at the same Adam step
    b[0].train_step(x[:B], cls[:B], reg[:B], 1e-3)
    for _ in range(3):
        idx = np.stack([rng.permutation(rows)[:B] for _ in widths])
        la = sl.mlp_train_rows(a, x, cls, reg, idx, 1e-3)
        lb = [m.train_step(x[i], cls[i], reg[i], 1e-3) for m, i in zip(b, idx)]
        assert la == lb
    ya, pa, ea = sl.mlp_forward_all(a, x[:B])
    for k, (p, q) in enumerate(zip(a, b)):
        assert bits_equal(p.get_params(), q.get_params()), k
        for got, want in zip((ya[k], pa[k], ea[k]), q.forward(x[:B])):
            assert bits_equal(got, want), k
    for m in a + b:
        m.close()


def test_the_same_net_twice_and_errors():
    rng = np.random.default_rng(0)
    x = rng.standard_normal((32, 21)).astype(np.float32)
    cls, reg = np.zeros(32, np.int32), rng.standard_normal((32, 6)).astype(np.float32)
    idx = np.stack([np.arange(16), np.arange(16, 32)])
    with sl.MLP(21, 9, 64, 32, seed=1) as m, sl.MLP(21, 9, 64, 32, seed=1) as q:
        la = sl.mlp_train_rows([m, m], x, cls, reg, idx, 1e-3)
        assert la == [q.train_step(x[i], cls[i], reg[i], 1e-3) for i in idx]
        assert bits_equal(m.get_params(), q.get_params())
        w = m.get_params()
        for bad in (dict(idx=idx + 1), dict(idx=idx - 1), dict(lr=0.0), dict(cls=cls + 3),
                    dict(idx=np.zeros((2, 33), np.int64))):
            with pytest.raises(sl.SpacelabError):
                sl.mlp_train_rows([m, q], **{**dict(x=x, cls=cls, reg=reg, idx=idx, lr=1e-3), **bad})
        assert bits_equal(m.get_params(), w)
