"""The fast sweep's reciprocal square root by gravity's share of a tile: lattices whose
largest share of gravity in a pair's force lies below, about and above 2^-31 (where the
unrefined root serves), against the same sums in extended precision.

Tolerance: a pair's factor carries 2.2e-15 (the reciprocal's 48.7 bits), a few roundings of
the algebra in front of it (s t)^-2 multiplies (4 x 1.1e-16 x 4) and the sums of up to 200
terms that are rounded relative to the largest partial sum (200 x 1.1e-16 at worst): 3e-14 of
the sum of the terms' sizes."""
import numpy as np
import pytest

import spacelab_amd as sl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("share", [-45, -34, -32, -31, -30, -20, 0, 10])
@pytest.mark.parametrize("n", [2, 130, 200])
def test_gravity_share(n, share):
    rng = np.random.default_rng(1000 * n + share)
    R = rng.uniform(0.9e-5, 1.1e-5, n)
    m = 2.25 * 4 / 3 * np.pi * R ** 3 * rng.uniform(0.9, 1.1, n)
    k = int(np.ceil(n ** (1 / 3)))
    cell = np.stack([np.arange(n) % k, np.arange(n) // k % k, np.arange(n) // k ** 2], 1)
    x = cell + rng.uniform(-.1, .1, (n, 3))
    p = sl.calibrate(sl.preset("config"), R, m, velocity=1.0, cor=0.64).replace(order=sl.ORDER_FAST)
    C = p.Ha / 6 * 64
    span = np.linalg.norm(x.max(0) - x.min(0))
    gq = (p.G * m ** 2 / (C * R ** 6)).max()
    x *= max((2.0 ** share / gq) ** 0.2 / span, 3e-5)     # the spheres stay apart
    with sl.Collider(n, p) as c:
        c.upload(sl.BallGroup(x, np.zeros((n, 3)), np.zeros((n, 3)), R, m, 0.4 * m * R ** 2))
        c.init_conditions()
        acc = c.download().acc
    L = np.longdouble
    x, R, m = x.astype(L), R.astype(L), m.astype(L)
    d = x[None] - x[:, None]
    d2 = (d ** 2).sum(-1)
    np.fill_diagonal(d2, 1)
    s = d2 - (R[None] + R[:, None]) ** 2
    t = d2 - (R[None] - R[:, None]) ** 2
    f = L(p.Ha) / 6 * 64 * (R[None] * R[:, None]) ** 3 / (s * t) ** 2 + L(p.G) * m[None] * m[:, None] / d2 ** L(1.5)
    np.fill_diagonal(f, 0)
    terms = f[..., None] * d
    ref = terms.sum(1) / m[:, None]
    size = np.abs(terms).sum(1) / m[:, None]
    assert (np.abs(acc - ref) <= 3e-14 * size).all(), float((np.abs(acc - ref) / size).max())


@pytest.mark.parametrize("ratio", [1e12, 1e13, 1e16])
def test_gravity_share_of_bodies_far_larger_than_the_median(ratio):
    """64 bodies (a block of their own) of `ratio` median radii, held by gravity alone: the
    median of 128 grains sets the scaled binary32 weights, which overflow at 7e12.  Same
    tolerance; the bodies lie 10 to 70 radii apart, inside the padding slots' distance."""
    big = 64
    R = np.concatenate([np.full(128, 1e8 / ratio), np.full(big, 1e8)])
    m = 2.25 * 4 / 3 * np.pi * R ** 3
    rng = np.random.default_rng(7)
    cell = np.stack(np.meshgrid(*[np.arange(4)] * 3, indexing="ij"), -1).reshape(-1, 3)
    grain = np.stack(np.meshgrid(np.arange(8), np.arange(4), np.arange(4), indexing="ij"), -1).reshape(-1, 3)
    x = np.concatenate([grain * 10 * R[0], 2e10 + (cell + rng.uniform(-.1, .1, (big, 3))) * 1.5e9])
    n = len(R)
    p = sl.preset("config").replace(order=sl.ORDER_FAST, kin=1.0, kout=0.64, dt=1e-9)
    with sl.Collider(n, p) as c:
        c.upload(sl.BallGroup(x, np.zeros((n, 3)), np.zeros((n, 3)), R, m, 0.4 * m * R ** 2))
        c.init_conditions()
        acc = c.download().acc[128:]
    L = np.longdouble
    d = x.astype(L)[None] - x.astype(L)[128:, None]
    d2 = (d ** 2).sum(-1)
    d2[np.arange(big), 128 + np.arange(big)] = 1
    terms = (L(p.G) * m.astype(L)[None] / d2 ** L(1.5))[..., None] * d
    ref, size = terms.sum(1), np.abs(terms).sum(1)
    assert (np.abs(acc - ref) <= 3e-14 * size).all(), float((np.abs(acc - ref) / size).max())
