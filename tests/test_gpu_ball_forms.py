"""The per-ball kernel's near pairs and slots where its forms change.  A lone near pair goes
through the fast engine in the reference's arithmetic, so its bits are the ordered pass's: in
the touching arm, in the band below h_min that does not touch, and with operands outside the
range of the arms' short divisions.  Systems around one batch of slots (80 blocks), where the
tiles begin to mark the slots that have near pairs, and around six batches (480 blocks), where
the next marks are read: eight wavefronts against four, which read every mask, bit for bit."""
import numpy as np
import pytest

from conftest import bits_equal

import spacelab_amd as sl

pytestmark = pytest.mark.gpu

FIELDS = ("pos", "vel", "w", "acc", "aacc", "velh", "wh")


def _run(g, p, steps, split=0, waves=0):
    with sl.Collider(g.num_particles, p) as c:
        if split:
            c.set_option("tile_split", split)
        if waves:
            c.set_option("ball_waves", waves)
        c.upload(g)
        e = [c.init_conditions()] + c.step(steps, 2)
        return c.download(), e


@pytest.mark.parametrize("scale", [1.0, 2.0 ** -110])
@pytest.mark.parametrize("flip", [False, True])
@pytest.mark.parametrize("kind", ["touch", "rest", "deep", "band", "heavy"])
def test_lone_near_pair_is_the_ordered_pass(kind, flip, scale):
    rng = np.random.default_rng(5)
    R = np.array([1e-5, 1.3e-5]) * scale
    m = np.array([1e-14, 2e-14])
    h_min = 1e-8 * scale
    gap = {"touch": -1e-3, "rest": -1e-3, "deep": -0.5, "band": 3e-4, "heavy": -1e-3}[kind]
    d = np.array([0.6, -0.48, 0.64]) * R.sum() * (1 + gap)
    if kind == "heavy":
        m = m * 2.0 ** 340
    v = np.zeros((2, 3)) if kind == "rest" else rng.standard_normal((2, 3)) * 1e-3 * scale
    w = np.zeros((2, 3)) if kind == "rest" else rng.standard_normal((2, 3))
    g = sl.BallGroup(np.array([[0, 0, 0], d]), v, w, R, m, 0.4 * m * R * R)
    if flip:
        g = sl.BallGroup(g.pos[::-1].copy(), v, w, R[::-1].copy(), m[::-1].copy(), g.moi[::-1].copy())
    p = sl.calibrate(sl.preset("config"), np.full(2, 1e-5), np.full(2, 1e-14), velocity=0.36301555459799423, cor=0.64)
    p = p.replace(h_min=max(h_min, 4e-4 * R.sum()))
    # elsewhere the first step takes the pair apart: its forces only
    steps = 4 if scale == 1.0 and kind in ("touch", "rest", "band") else 0
    a, ea = _run(g, p.replace(order=sl.ORDER_FAST), steps)
    b, eb = _run(g, p, steps)
    for f in FIELDS:
        assert bits_equal(getattr(a, f), getattr(b, f)), f
    assert [e.contacts for e in ea] == [e.contacts for e in eb]
    assert ea[0].contacts == (0 if kind == "band" else 1)
    for x, y in zip(ea, eb):
        assert bits_equal(np.float64(x.PE), np.float64(y.PE)) and bits_equal(np.float64(x.KE), np.float64(y.KE))


@pytest.mark.parametrize("precision", [sl.PREC_FP64, sl.PREC_MIXED])
@pytest.mark.parametrize("n", [5120, 5121, 30720, 30721])
def test_marked_slots_same_bits(n, precision):
    # a line of touching pairs and triples in shuffled order: every block has near pairs in its
    # own slot and, where the curve jumps, in others
    rng = np.random.default_rng(n)
    k = int(np.ceil(n ** (1 / 3)))
    cell = np.arange(n)
    x = np.stack([cell % k, cell // k % k, cell // k ** 2], 1) * 2.1e-5
    x[::3, 0] += 2e-6
    pos = x[rng.permutation(n)]
    R = np.full(n, 1e-5)
    m = 2.25 * 4 / 3 * np.pi * R ** 3
    g = sl.BallGroup(pos, rng.standard_normal((n, 3)) * 1e-3, rng.standard_normal((n, 3)), R, m, 0.4 * m * R * R)
    p = sl.calibrate(sl.preset("config"), R, m, velocity=0.36301555459799423, cor=0.64)
    p = p.replace(order=sl.ORDER_FAST, precision=precision)
    a, ea = _run(g, p, 3, 1, 8)
    b, eb = _run(g, p, 3, 1, 4)
    assert ea[0].contacts > n // 4
    for f in FIELDS:
        assert bits_equal(getattr(a, f), getattr(b, f)), f
    assert [x.as_array().tobytes() for x in ea] == [x.as_array().tobytes() for x in eb]
    assert [x.contacts for x in ea] == [x.contacts for x in eb]


@pytest.mark.parametrize("n", [5121, 5185, 5249, 5313])
@pytest.mark.parametrize("queue", [1, 2])
def test_grouped_rows(n, queue):
    """81 to 84 blocks: rows whose last group of four tiles has every length.  One and two
    wavefronts a tile add the i sides of four and two tiles before they are stored, four
    wavefronts keep every tile's: sums of at most 84 x 64 terms in another order, each rounded
    once (1.1e-16) on at most the sum of the terms' sizes, which for these lattices is below 50
    times the largest acceleration: 84 x 64 x 1.1e-16 x 50 = 3e-11 at the very worst, and
    sqrt of the count in practice: 1e-12 of the largest."""
    rng = np.random.default_rng(n)
    k = int(np.ceil(n ** (1 / 3)))
    cell = rng.permutation(k ** 3)[:n]
    pos = (np.stack([cell % k, cell // k % k, cell // k ** 2], 1) + rng.uniform(-.05, .05, (n, 3))) * 2.5e-5
    R = np.full(n, 1e-5)
    m = 2.25 * 4 / 3 * np.pi * R ** 3
    zero = np.zeros((n, 3))
    g = sl.BallGroup(pos, zero, zero.copy(), R, m, 0.4 * m * R * R)
    p = sl.calibrate(sl.preset("config"), R, m, velocity=0.36301555459799423, cor=0.64).replace(order=sl.ORDER_FAST)
    acc = []
    for split in (4, 2, 1):
        with sl.Collider(n, p) as c:
            c.set_option("tile_split", split)
            c.set_option("tile_queue", queue)
            c.upload(g)
            c.init_conditions()
            acc.append(c.download().acc)
    top = np.abs(acc[0]).max()
    assert np.abs(acc[1] - acc[0]).max() <= 1e-12 * top and np.abs(acc[2] - acc[0]).max() <= 1e-12 * top
