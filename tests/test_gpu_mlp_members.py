"""Several nets through shared launches against the same nets one by one: the sums are the
same, so every comparison is of bits.  Nets laid out alike share launches, up to 16 of them;
nets of different widths or largest batch, in the layer form, or the same net twice go one by
one."""
import functools

import numpy as np
import pytest

from conftest import bits_equal

import spacelab_amd as sl
from oracle.mlp import bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("widths,n_in,n_out,B,max_batch", [
    ([256] * 4, 21, 9, 256, [256] * 4), ([256], 21, 9, 33, [40]), ([64] * 17, 21, 9, 17, [17] * 17), ([48] * 16, 40, 40, 1, [3] * 16),
    ([64] * 3, 21, 9, 16, [32] * 3), ([64] * 3, 21, 9, 16, [31] * 3), ([256, 256, 80], 21, 9, 40, [64] * 3), ([64] * 2, 21, 9, 40, [64, 80]), ([528] * 2, 21, 9, 40, [40] * 2)])
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
    for steps in (1, 2, 5):
        idx = np.stack([[rng.permutation(rows)[:B] for _ in widths] for _ in range(steps)])
        la = sl.mlp_train_rows(a, x, cls, reg, idx, 1e-3)
        lb = [[m.train_step(x[i], cls[i], reg[i], 1e-3) for m, i in zip(b, step)] for step in idx]
        assert la.tolist() == lb
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
        la = sl.mlp_train_rows([m, m], x, cls, reg, idx[None], 1e-3)
        assert la.tolist() == [[q.train_step(x[i], cls[i], reg[i], 1e-3) for i in idx]]
        idx = np.stack([idx, idx[::-1]])
        assert bits_equal(m.get_params(), q.get_params())
        w = m.get_params()
        for bad in (dict(idx=idx + 1), dict(idx=idx - 1), dict(lr=0.0), dict(cls=cls + 3),
                    dict(idx=np.zeros((2, 2, 33), np.int64))):
            with pytest.raises(sl.SpacelabError):
                sl.mlp_train_rows([m, q], **{**dict(x=x, cls=cls, reg=reg, idx=idx, lr=1e-3), **bad})
        assert bits_equal(m.get_params(), w)


@pytest.mark.parametrize("members,max_batch,rows", [(4, 64, 0), (4, 64, 1), (4, 64, 32), (4, 64, 33), (4, 64, 97), (1, 1, 3), (16, 2, 5),
                                                    (2, 3, 7), (3, 4096, 5000)])
def test_ensemble_is_the_members_mean(members, max_batch, rows):
    """Normalising, the sums over the members and the choice are the same operations as in
    numpy, so the same bits; the entropy's logarithm may differ by an ulp or two."""
    rng = np.random.default_rng(members + rows)
    X = rng.standard_normal((rows, 21)) * 3 + 1
    if rows > 4:
        X[2, 5] = np.nan
        X[3, 0] = 1e300
    mean, std = rng.standard_normal(21), rng.uniform(0.5, 2, 21)
    nets = [sl.MLP(21, 9, 80, max_batch, seed=k) for k in range(members)]
    assert sl.mlp_alike(nets) and not sl.mlp_alike(nets + nets[:1])
    cls, reg, prob, ent = sl.mlp_ensemble(nets, X, mean, std)
    P, Y = np.zeros((rows, 3)), np.zeros((rows, 6))
    with np.errstate(over="ignore", invalid="ignore"):
        Xn = np.ascontiguousarray((X - mean) / std, dtype=np.float32)
        for m in nets:
            for k in range(0, rows, max_batch):
                y, p, _ = m.forward(Xn[k:k + max_batch])
                P[k:k + len(p)] += p
                Y[k:k + len(y)] += y[:, 3:]
        P /= members
        Y /= members
        want = -(P * np.log(np.where(P > 0, P, 1.0))).sum(1)
    assert bits_equal(cls, P.argmax(1).astype(np.int32))
    assert np.array_equal(reg, Y.astype(np.float32), equal_nan=True) and np.array_equal(prob, P, equal_nan=True)
    assert np.allclose(ent, want, rtol=0, atol=1e-15 * 8, equal_nan=True)
    for m in nets:
        m.close()


@functools.lru_cache
def _forms():
    X = np.random.default_rng(3).standard_normal((37, 21)) * 2 + 0.3
    f32 = lambda a: a.astype(np.float32)
    # rows whose normalising rounds to other bfloat16 inputs in binary32 than in binary64
    rng = np.random.default_rng(4)
    mean, std = rng.standard_normal(21), rng.uniform(0.5, 2, 21)
    Z = f32(rng.standard_normal((300000, 21)))
    edge = Z[(bf16((Z - f32(mean)) / f32(std)) != bf16(f32((Z.astype(float) - f32(mean)) / f32(std)))).any(1)]
    assert len(edge) > 5
    return {"binary32 where it differs": (edge, f32), "halves": (X.astype(np.float16), f32),
            "binary32 rows and mean": (edge, (f32, lambda a: a)),
            "rows": (X, None), "fortran": (np.asfortranarray(X), None), "every other": (np.repeat(X, 2, 0)[::2], None),
            "reversed": (X[::-1, ::-1], None), "integers": ((10 * X).astype(np.int64), None), "list": (X.tolist(), None),
            "binary32 rows": (f32(X), None), "binary32 throughout": (f32(X), f32), "binary32 statistics": (X, f32),
            "extended": (X.astype(np.longdouble), None), "one column": (X[:, :1], None), "one row's statistics": (X, lambda a: a[None]),
            "scalar statistics": (X, lambda a: a[0]), "scalar for binary32 rows": (f32(X), lambda a: float(a[0])), "none": (X[:0], None)}


@pytest.mark.parametrize("form", list(_forms()))
def test_predict_takes_every_form_of_rows(form):
    """Rows and statistics of any shape, order and type that numpy normalises: the same bits as
    normalising them there and averaging the nets one by one."""
    from spacelab_amd import surrogate as S
    X, change = _forms()[form]
    rng = np.random.default_rng(4)
    mean, std = rng.standard_normal(21), rng.uniform(0.5, 2, 21)
    s = S.Surrogate(width=64, n_models=3, max_batch=16)
    change = change if isinstance(change, tuple) else (change, change)
    s.norm = S.Normaliser(*(a if c is None else c(a) for c, a in zip(change, (mean, std))))
    Xn = np.ascontiguousarray((X - s.norm.mean) / s.norm.std, dtype=np.float32)
    P, Y = np.zeros((len(Xn), 3)), np.zeros((len(Xn), S.N_REG))
    for m in s.mlps:
        for k in range(0, len(Xn), 16):
            y, p, _ = m.forward(Xn[k:k + 16])
            P[k:k + len(p)] += p
            Y[k:k + len(y)] += y[:, 3:]
    P, Y = P / 3, Y / 3
    cls, reg, prob, ent = s.predict(X)
    assert bits_equal(cls, P.argmax(1)) and bits_equal(reg, Y.astype(np.float32)) and bits_equal(prob, P)
    assert np.allclose(ent, -(P * np.log(np.where(P > 0, P, 1.0))).sum(1), rtol=0, atol=1e-15 * 8)
    s.close()


def test_predict_refuses_nets_of_other_outputs_or_smaller_batches():
    from spacelab_amd import surrogate as S
    X = np.zeros((40, 21))
    for nets, error in (([sl.MLP(21, 8, 64, 64, k) for k in range(2)], ValueError),
                        ([sl.MLP(21, 9, 64, 32, k) for k in range(2)], sl.SpacelabError)):
        s = S.Surrogate(max_batch=64, mlps=nets)
        s.norm = S.Normaliser(np.zeros(21), np.ones(21))
        with pytest.raises(error):
            s.predict(X)
        s.close()


def test_fit_takes_labels_in_a_column():
    from spacelab_amd import surrogate as S
    rng = np.random.default_rng(5)
    X, cls, reg = rng.standard_normal((64, 21)), rng.integers(0, 3, 64), rng.standard_normal((64, 6))
    a, b = (S.Surrogate(width=64, n_models=2, max_batch=32) for _ in range(2))
    assert a.fit(X, cls, reg, epochs=2, batch=32) == b.fit(X, cls[:, None], reg.reshape(64, 2, 3), epochs=2, batch=32)
    for p, q in zip(a.mlps, b.mlps):
        assert bits_equal(p.get_params(), q.get_params())
    for short in (dict(cls=cls[:40]), dict(reg=reg[:40])):
        with pytest.raises(IndexError):
            a.fit(X, **{**dict(cls=cls, reg=reg), **short}, epochs=1, batch=32)
    a.close()
    b.close()
