"""The direct sum's FP64 pair term bit for bit, and its source groups at their
edges, against the oracle.

A system of two bodies has one term, so its FP64 accelerations are the
oracle's exactly: every quotient and root correctly rounded, over scales and
softenings inside and outside the fast form's range, with zero offsets and
mantissas of all ones among them. Larger systems sum the same terms in groups:
n 2^-53 times the sum of the terms' magnitudes bounds the difference of two
orders of summation. Mixed precision: terms in FP32, 1e-6 of that sum."""
import numpy as np
import pytest

import physim_amd as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def bodies(pos, mass):
    s = np.zeros(len(pos), P.ENTITY)
    for a, f in enumerate("xyz"):
        s[f] = pos[:, a]
    s["mass"] = mass
    s["radius"] = 0.01
    return s


@pytest.mark.parametrize("scale,mass,e", [
    (1.0, 1.0, 0.5), (1.0, 1e5, 0.01), (1e-3, 1e-6, 0.0), (1e6, 1e30, 1.0),
    (1e-90, 1.0, 0.0), (1e120, 1.0, 1e-3), (1.0, 1e-320, 0.5), (3e-107, 1.0, 0.0),
    (1e-140, 1.0, 0.0), (1e140, 1.0, 0.0), (1.0, 1e95, 0.5)])
def test_one_term_bit_exact(engine, scale, mass, e):
    rng = np.random.default_rng(int(abs(np.log10(scale)) * 7 + abs(np.log10(mass))))
    states = []
    ones = np.nextafter(2.0, 0.0)
    for k in range(200):
        p = rng.uniform(-1.0, 1.0, (2, 3)) * scale
        if k % 5 == 1:
            p[1, :2] = p[0, :2]  # offsets of zero
        if k % 5 == 2:
            p = np.array([[0.0, 0.0, 0.0], [ones, 0.0, 0.0]]) * scale * 2.0 ** (k % 7)
        if k % 5 == 3:
            p = np.rint(p / scale * 8) / 8 * scale  # short mantissas, equal places
        states.append(bodies(p, mass * rng.uniform(0.5, 2.0, 2)))
    sims = [P.Sim(engine, s, kind="simple_astro", precision="fp64", e=e) for s in states]
    for sim, s in zip(sims, states):
        a = sim.accel()
        np.testing.assert_array_equal(a, O.simple_transform(s, e))
        sim.close()


@pytest.mark.parametrize("n", [256, 257, 1024, 1025, 1537, 4097, 8195, 18900, 19200])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_source_groups(engine, n, precision):
    rng = np.random.default_rng(n)
    s = bodies(rng.uniform(-1.0, 1.0, (n, 3)), rng.uniform(0.5, 1.5, n) / n)
    sim = P.Sim(engine, s, kind="simple_astro", precision=precision, e=0.1)
    a = sim.accel()
    rows = np.unique(np.concatenate([np.arange(0, n, max(1, n // 97)), [n - 1]]))
    ref = O.simple_transform_rows(s, 0.1, rows)
    pos = np.stack([s["x"], s["y"], s["z"]], 1)
    r2 = ((pos[rows, None] - pos[None]) ** 2).sum(-1)
    size = (s["mass"] / (r2 + 0.1)).sum(1)  # the sum of the terms' magnitudes
    bound = (n * 2.0 ** -53 if precision == "fp64" else 1e-6) * size
    assert (np.abs(a[rows] - ref).max(1) <= bound).all()
    # alone, in a batch and through the allocation-free call: the same bits
    small = bodies(rng.uniform(-1.0, 1.0, (300, 3)), np.full(300, 1.0 / 300))
    kw = dict(kind="simple_astro", precision=precision, e=0.1, dt=1e-4)
    pair = [P.Sim(engine, x, **kw) for x in (small, s)]
    engine.batch_step(pair, 2)
    one = P.Sim(engine, s, **kw)
    one.step(2)
    np.testing.assert_array_equal(pair[1].download(), one.download())
    b = engine.transform_noalloc(s, kind="simple_astro", e=0.1, precision=precision)
    np.testing.assert_array_equal(b.view(np.float64).reshape(n, 3), a)
    for x in pair + [one, sim]:
        x.close()


@pytest.mark.parametrize("n", [1, 255, 257, 700])
def test_energy_groups(engine, n):
    """Energy terms summed in groups against the oracle's: (n + 1000) 2^-53
    of the sum of their magnitudes."""
    rng = np.random.default_rng(n)
    s = bodies(rng.uniform(-1.0, 1.0, (n, 3)), rng.uniform(0.5, 1.5, n) / n)
    for f in ("vx", "vy", "vz"):
        s[f] = rng.normal(size=n)
    sim = P.Sim(engine, s, kind="simple_astro", e=0.1)
    got = sim.energy()
    ref = np.asarray(O.energy(s, 0.1))
    speed = np.sqrt(s["vx"] ** 2 + s["vy"] ** 2 + s["vz"] ** 2)
    size = np.array([abs(ref[0]), abs(ref[1]), abs(ref[0]) + abs(ref[1])] +
                    [float((s["mass"] * speed).sum())] * 3)
    assert (np.abs(got - ref[:6]) <= (n + 1000) * 2.0 ** -53 * size).all()
    sim.close()


@pytest.mark.parametrize("ma,mb", [
    (1e-150, 1e-150), (1.0, 1e-300), (1e-300, 1e10), (2.0 ** -181, 2.0 ** -179), (0.0, 1.0),
    (2.0 ** 199, 2.0 ** 201), (2.0 ** 290, 2.0 ** 290), (1e-155, 3e-155)])
@pytest.mark.parametrize("scale,tiny,e", [
    (1.0, 0.0, 0.5), (1.0, 1e-295, 0.5), (1.0, 3e-310, 0.0), (1e-8, 2.0 ** -301, 1e-30),
    (2.0 ** 99, 2.0 ** -300, 0.0), (2.0 ** 101, 0.0, 1.0), (2.0 ** -301, 0.0, 0.0),
    (2.0 ** -299, 0.0, 0.0)])
def test_one_term_at_the_ends_of_the_range(engine, ma, mb, scale, tiny, e):
    """Masses, separations and single components of one near and past the ends
    of the fast form's range: the oracle's bits (infinities and NaN where it
    has them), in the direct sum, and in the walk where the two bodies are far
    enough apart for a tree."""
    rng = np.random.default_rng(7)
    for k in range(24):
        p = rng.uniform(0.5, 1.0, (2, 3)) * scale * [[-1.0], [1.0]]
        if tiny or k % 3 == 0:
            p[:, k % 3] = rng.uniform(-1.0, 1.0, 2) * tiny
        s = bodies(p, [ma * rng.uniform(0.9, 1.1), mb * rng.uniform(0.9, 1.1)])
        sim = P.Sim(engine, s, kind="simple_astro", precision="fp64", e=e)
        np.testing.assert_array_equal(sim.accel(), O.simple_transform(s, e))
        sim.close()
        if 1e-8 <= scale <= 1.0:
            ref, _, fault = O.bh_transform(s, 0.0, e)
            assert fault == 0
            sim = P.Sim(engine, s, kind="astro2", precision="fp64", theta=0.0, e=e)
            np.testing.assert_array_equal(sim.accel(), ref)
            sim.close()


def test_range_is_looked_at_for_every_source(engine):
    """One source outside the range among 700: the sum of each body's terms in
    source order, as one block sums them (n 2^-53 of the terms' magnitudes)."""
    rng = np.random.default_rng(11)
    for at in (0, 255, 256, 699):
        s = bodies(rng.uniform(-1.0, 1.0, (700, 3)) * 1e-100, np.full(700, 1e-200))
        s["mass"][at] = 1e-60
        s["x"][at] = 1e-120
        sim = P.Sim(engine, s, kind="simple_astro", precision="fp64", e=1e-190)
        a = sim.accel()
        ref = O.simple_transform(s, 1e-190)
        pos = np.stack([s["x"], s["y"], s["z"]], 1)
        r2 = ((pos[:, None] - pos[None]) ** 2).sum(-1)
        size = (s["mass"] / (r2 + 1e-190)).sum(1)
        assert np.isfinite(ref).all()
        assert (np.abs(a - ref).max(1) <= 700 * 2.0 ** -53 * size).all()
        sim.close()
