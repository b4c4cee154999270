"""The ordered pair pass where its special paths begin, every launch shape bitwise against the
oracle: systems in which nearly every pair touches (more touching pairs than the contact table,
a batch's kept steps and a ball's 64 slots hold), and radii, masses, distances and parameters
outside the exponent range of the far arm's square root and divisions (the general arm takes
those pairs).  Runs of every length from 1 to 5, so that odd and even runs of graphs occur."""
import numpy as np
import pytest

from conftest import bits_equal

import spacelab_amd as sl

pytestmark = pytest.mark.gpu


def _group(rng, n, spread, r=1e-5, v=1e-3):
    pos = rng.uniform(-spread, spread, (n, 3)) * r
    R = r * rng.uniform(0.8, 1.2, n)
    m = 2.25 * 4 / 3 * np.pi * R ** 3
    return sl.BallGroup(pos, v * rng.standard_normal((n, 3)), 10 * rng.standard_normal((n, 3)), R, m, 0.4 * m * R * R)


def _case(name):
    rng = np.random.default_rng(sum(map(ord, name)))
    kw = {}
    if name == "dense-131":          # almost all pairs touch
        g = _group(rng, 131, 0.8)
    elif name == "dense-70":
        g = _group(rng, 70, 1.5)
    elif name == "two":              # one pair, touching
        g = _group(rng, 2, 0.3)
    elif name == "tiny-radius":      # one partner below the radius range
        g = _group(rng, 90, 30)
        g.R[40] = 1e-33
    elif name == "huge-mass":
        g = _group(rng, 67, 30)
        g.m[3] = 1e95
        g.moi[3] = 1e85
    elif name == "far-away":         # distances above the range, and coordinates that cancel to 0
        g = _group(rng, 66, 30)
        g.pos[65] = [3e31, 0, 0]
        g.pos[7] = g.pos[8] + [0, 0, 4e-5]
    elif name == "small-units":      # every radius, and h_min, below the range
        g = _group(rng, 65, 20, r=1e-33, v=0.0)
        g.m[:] = 1e-30
        g.moi[:] = 1e-95
        kw = dict(h_min=1e-34, dt=1e-120)
    elif name == "no-gravity":
        g = _group(rng, 129, 12)
        kw = dict(G=0.0)
    return g, kw


@pytest.mark.parametrize("name", ["dense-131", "dense-70", "two", "tiny-radius", "huge-mass", "far-away", "small-units",
                                  "no-gravity"])
def test_special_paths_bitwise(oracle_mod, name):
    g, kw = _case(name)
    p = sl.calibrate(sl.preset("config"), np.full(4, 1e-5), np.full(4, 1e-14), velocity=0.36301555459799423, cor=0.64)
    p = p.replace(**kw)
    P = oracle_mod.Params(G=p.G, Ha=p.Ha, h_min=p.h_min, u_s=p.u_s, u_r=p.u_r, kin=p.kin, kout=p.kout, dt=p.dt,
                          far_gravity=p.far_gravity)
    n = g.num_particles
    for steps in (1, 2, 3, 5):
        s, _, _ = oracle_mod.run(oracle_mod.State(g.pos, g.vel, g.w, g.R, g.m, g.moi), P, steps + 1, 0, mode="gather")
        assert np.isfinite(s.acc).all() and np.isfinite(s.aacc).all()
        for shape in range(1, 10):
            with sl.Collider(n, p) as c:
                c.set_option("ordered_shape", shape)
                c.upload(g)
                c.init_conditions()
                if steps > 2:
                    c.step(1)           # the first step of a context is launched directly
                    c.step(steps - 1)
                else:
                    c.step(steps)
                out = c.download()
            for k in ("pos", "vel", "velh", "w", "wh", "acc", "aacc"):
                assert bits_equal(getattr(out, k), getattr(s, k)), (name, steps, shape, k)


def test_contacts_counted_on_every_path():
    """Touching pairs counted once each, from the table and where they are met: every shape
    reports the number of overlapping pairs."""
    g, _ = _case("dense-131")
    p = sl.calibrate(sl.preset("config"), g.R, g.m, velocity=0.36301555459799423, cor=0.64)
    d = np.linalg.norm(g.pos[:, None] - g.pos[None], axis=2)
    want = int(np.triu(d < g.R[:, None] + g.R[None], 1).sum())
    after = []
    for shape in range(1, 10):
        with sl.Collider(131, p) as c:
            c.set_option("ordered_shape", shape)
            c.upload(g)
            assert c.init_conditions().contacts == want
            after.append(c.step(1, 1)[0].contacts)
    assert len(set(after)) == 1 and abs(after[0] - want) < 0.01 * want, after


@pytest.mark.parametrize("n,at", [(66, 0), (150, 75), (150, 149), (270, 131)])
def test_a_ball_with_contacts_all_over_bitwise(oracle_mod, n, at):
    """One large sphere that all others touch, first, last or between: every batch of its
    workgroup has touching pairs at every step, more than the contact table holds."""
    k = np.arange(n - 1) + 0.5
    polar, turn = np.arccos(1 - 2 * k / (n - 1)), np.pi * (1 + 5 ** 0.5) * k
    u = np.stack([np.cos(turn) * np.sin(polar), np.sin(turn) * np.sin(polar), np.cos(polar)], 1)
    R = np.concatenate([[1e-5 * np.sqrt(0.4 * n)], np.full(n - 1, 1e-5)])
    pos = np.concatenate([[[0, 0, 0]], u * (R[0] + 0.999e-5)])
    order = np.roll(np.arange(n), at)
    rng = np.random.default_rng(n + at)
    pos, R = np.ascontiguousarray(pos[order]), R[order]
    m = 2.25 * 4 / 3 * np.pi * R ** 3
    g = sl.BallGroup(pos, 1e-3 * rng.standard_normal((n, 3)), 10 * rng.standard_normal((n, 3)), R, m, 0.4 * m * R * R)
    p = sl.calibrate(sl.preset("config"), R, m, velocity=0.36301555459799423, cor=0.64)
    P = oracle_mod.Params(G=p.G, Ha=p.Ha, h_min=p.h_min, u_s=p.u_s, u_r=p.u_r, kin=p.kin, kout=p.kout, dt=p.dt,
                          far_gravity=p.far_gravity)
    s, _, _ = oracle_mod.run(oracle_mod.State(g.pos, g.vel, g.w, g.R, g.m, g.moi), P, 6, 0, mode="gather")
    touching = int(np.triu(np.linalg.norm(pos[:, None] - pos[None], axis=2) < R[:, None] + R[None], 1).sum())
    assert touching >= n - 1
    for shape in range(1, 10):
        with sl.Collider(n, p) as c:
            c.set_option("ordered_shape", shape)
            c.upload(g)
            assert c.init_conditions().contacts == touching
            c.step(1)
            c.step(4)
            out = c.download()
        for f in ("pos", "vel", "velh", "w", "wh", "acc", "aacc"):
            assert bits_equal(getattr(out, f), getattr(s, f)), (shape, f)
