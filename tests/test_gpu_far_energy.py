"""Potential energy of far pairs in the fast engine, on lattices of separate spheres.

The engine takes the van der Waals energy of a pair from a series in y = 4 Ri Rj / (d^2 - (Ri -
Rj)^2) for y <= 1/8 and from the closed form above; spacings of 5.4 to 5.9 radii put pairs on
both sides of the line, 3, 8 and 40 radii nearly all on one.  The expected sum is the same series
(to 80 terms) or the closed form in extended precision, added exactly.

Tolerance 1e-13: a series term carries a few ulps of 1.1e-16, the closed form at y > 1/8 loses
at most 6/y^2 ulps (4e-14) of a pair that weighs y^3, and the sum of at most 8385 equal-signed
terms in a tree of 64 adds fewer than 100 ulps (1.1e-14)."""
import math

import numpy as np
import pytest

import spacelab_amd as sl

pytestmark = pytest.mark.gpu


def _expected(pos, R, Ha):
    out = []
    for i in range(len(R)):
        d2 = ((pos[:i] - pos[i]) ** 2).sum(1)
        for j in range(i):
            y = 4 * R[i] * R[j] / (d2[j] - (R[i] - R[j]) ** 2)
            if y < 0.4:
                u = y ** 3 * math.fsum((0.5 - 1 / k) * y ** (k - 3) for k in range(3, 80))
            else:
                z = np.longdouble(y)
                u = float(z / 2 / (1 - z) + z / 2 + np.log1p(-z))
            out.append(-Ha / 6 * u)
    return math.fsum(out)


@pytest.mark.parametrize("precision", [sl.PREC_FP64, sl.PREC_MIXED])
@pytest.mark.parametrize("spacing,n", [(3.0, 130), (5.4, 65), (5.66, 130), (5.9, 64), (7.6, 65), (8.0, 130), (8.4, 64), (40.0, 130), (40.0, 2)])
def test_far_pair_energy(spacing, n, precision):
    rng = np.random.default_rng(int(spacing * 10) + n)
    side = math.ceil(n ** (1 / 3))
    grid = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    r = 1e-5
    R = r * rng.uniform(0.9, 1.1, n)
    pos = spacing * r * grid.astype(np.float64)
    m = 2.25 * 4 / 3 * math.pi * R ** 3
    zero = np.zeros((n, 3))
    g = sl.BallGroup(pos, zero, zero.copy(), R, m, 0.4 * m * R * R)
    p = sl.calibrate(sl.preset("reference"), R, m, velocity=0.36, cor=0.64)
    with sl.Collider(n, p.replace(order=sl.ORDER_FAST, precision=precision)) as c:
        c.upload(g)
        e = c.init_conditions()
    assert e.contacts == 0 and e.KE == 0.0
    want = _expected(pos, R, p.Ha)
    assert abs(e.PE - want) <= 1e-13 * abs(want)
