"""State read-back through the packing kernel: pieces of the staging buffer (6,208 balls of
seven vectors fill one), ragged systems across its pieces, engine and canonical order.
Values are copied, so every comparison is of bits."""
import numpy as np
import pytest

from conftest import bits_equal

import spacelab_amd as sl

pytestmark = pytest.mark.gpu

FIELDS = ("pos", "vel", "w", "acc", "aacc")


def _grid(n, seed):
    """n separate balls on a jittered lattice, in shuffled (not Morton) order."""
    rng = np.random.default_rng(seed)
    k = int(np.ceil(n ** (1 / 3)))
    cell = rng.permutation(k ** 3)[:n]
    R = rng.uniform(0.5e-5, 1e-5, n)
    m = 2.25 * 4 / 3 * np.pi * R ** 3
    pos = (np.stack([cell % k, cell // k % k, cell // k ** 2], 1) + rng.uniform(-.1, .1, (n, 3))) * 3e-5
    return sl.BallGroup(pos, rng.normal(size=(n, 3)), rng.normal(size=(n, 3)), R, m, 0.4 * m * R ** 2)


def _params(g, **kw):
    return sl.calibrate(sl.preset("config"), g.R, g.m, velocity=1.0, cor=0.64).replace(**kw)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 6208, 6209, 13001])
def test_collider_read_back(n):
    g = _grid(n, n)
    p = _params(g, order=sl.ORDER_FAST)
    with sl.Collider(n, p) as c:
        c.upload(g)
        out = c.download()
        for f in ("pos", "vel", "w"):
            assert bits_equal(getattr(out, f), getattr(g, f)), f
        c.init_conditions()
        c.step(2)
        engine = c.download()
        again = c.download()
        c.set_params(p)                       # brings the caller's order up to date
        canonical = c.download()
        for f in FIELDS + ("velh", "wh"):
            assert bits_equal(getattr(engine, f), getattr(canonical, f)), f
            assert bits_equal(getattr(engine, f), getattr(again, f)), f
        # any subset, the rest untouched
        half = np.full((n, 3), 7.0)
        c._check(sl.lib().sl_download_half(c._ctx, None, sl._dp(half)), "half")
        assert bits_equal(half, canonical.wh)
        assert not bits_equal(engine.pos, g.pos)


@pytest.mark.parametrize("sizes", [[1], [64, 1, 65, 127], [6000, 200, 1, 8, 9000, 64, 3], [7] * 1000])
def test_batch_read_back(sizes):
    groups = [_grid(n, 100 + k) for k, n in enumerate(sizes)]
    p = _params(groups[0], order=sl.ORDER_FAST)
    with sl.Batch(len(sizes), sum(sizes), p) as b:
        b.upload(groups)
        for g, o in zip(groups, b.download()):
            for f in ("pos", "vel", "w", "R", "m", "moi"):
                assert bits_equal(getattr(o, f), getattr(g, f)), f
        b.init_conditions()
        b.step(2)
        engine = b.download()
        b.set_system_params()                 # brings the caller's order up to date
        canonical = b.download()
        for g, e, o in zip(groups, engine, canonical):
            for f in FIELDS:
                assert bits_equal(getattr(e, f), getattr(o, f)), f
            assert not bits_equal(e.pos, g.pos)


def _root(a):
    while a.base is not None:
        a = a.base
    return a


def test_a_kept_group_does_not_keep_the_batch():
    """What one group of a batch, or one energy of many, holds in memory is its own or bounded."""
    sizes = [250] * 40 + [17000] + [3] * 30 + [8192, 8192, 1, 64]
    groups = [_grid(n, k) for k, n in enumerate(sizes)]
    with sl.Batch(len(sizes), sum(sizes), _params(groups[0], order=sl.ORDER_FAST)) as b:
        b.upload(groups)
        energies = b.init_conditions()
        for g, o in zip(groups, b.download()):
            assert o.num_particles == g.num_particles
            for f in ("pos", "vel", "w", "R", "m", "moi"):
                assert bits_equal(getattr(o, f), getattr(g, f)), f
            held = {id(r): r.nbytes for r in (_root(getattr(o, f)) for f in ("pos", "vel", "w", "R", "m", "moi", "acc", "aacc"))}
            assert sum(held.values()) <= 18 * 8 * max(32768, g.num_particles)
    assert all(_root(e.p).nbytes <= 24 * 1024 for e in energies)
    with sl.Collider(2, _params(_grid(2, 0), order=sl.ORDER_FAST)) as c:
        c.upload(_grid(2, 0))
        c.init_conditions()
        e = c.step(3000, 1)
    assert len(e) == 3000 and all(_root(x.p).nbytes <= 24 * 1024 and _root(x.L).nbytes <= 24 * 1024 for x in e)


def test_parts_that_do_not_hold_every_system_are_refused():
    import ctypes as C
    groups = [_grid(n, n) for n in (5, 70, 3)]
    with sl.Batch(3, 78, _params(groups[0], order=sl.ORDER_FAST)) as b:
        with pytest.raises(sl.SpacelabError):
            b.download()                      # nothing uploaded
        b.upload(groups)
        bufs = [np.empty((5, 78, 3)) for _ in range(3)]
        call = lambda *ns: sl.lib().sl_batch_download_parts(b._b, len(ns), (C.c_int * len(ns))(*ns),
                                                            (C.c_void_p * 3)(*(x.ctypes.data for x in bufs)))
        assert call(1, 2) == 0 and call(3) == 0 and call(1, 1, 1) == 0
        for bad in ((1, 1), (2, 2), (0, 3), (4,), (-1, 4), ()):
            assert call(*bad) < 0, bad
