"""The walk's two phases at their edges, against the oracle: wave and chunk
sizes, waves whose bodies are all fixed, opening tests that tie exactly (cells
whose half-width over distance equals theta), opening angles outside the
range the test's thresholds cover, and near fields.

Interaction counts are equal. FP64 accelerations: the node centres of mass
differ from the oracle's by their summation order only, n 2^-53 of the node's
coordinates at most, and a separation no shorter than 1e-4 of them turns that
into n 2^-53 1e4 of a term: 1e-9 of the largest acceleration at n < 1000.
Mixed: terms rounded to FP32 a few times each, 1e-6 of it."""
import numpy as np
import pytest

import physim_amd as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def cloud(n, seed):
    rng = np.random.default_rng(seed)
    s = np.zeros(n, P.ENTITY)
    for f in "xyz":
        s[f] = rng.uniform(-1.0, 1.0, n)
    s["mass"] = rng.uniform(0.5, 1.5, n) / n
    s["radius"] = 0.01
    return s


def lattice(m):
    """m^3 bodies on a lattice that the octree's cells cut evenly."""
    s = np.zeros(m ** 3, P.ENTITY)
    k = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)
    for a, f in enumerate("xyz"):
        s[f] = (k[:, a] - (m - 1) / 2) / 4
    s["mass"] = 1.0 / len(s)
    return s


def check(engine, s, theta, near=0.0, kind="astro2"):
    dim = 3 if kind == "astro2" else 2
    ref, counts, fault = (O.bh_transform_near(s, theta, 0.1, near, dim=dim, counts=True) if near
                          else O.bh_transform(s, theta, 0.1, dim=dim, counts=True))
    assert fault == 0
    big = np.abs(ref).max() + 1e-300
    for precision, bound in (("fp64", 1e-9), ("mixed", 1e-6)):
        for counting in (True, False):
            sim = P.Sim(engine, s, kind=kind, precision=precision, theta=theta, e=0.1)
            sim.set_near_field(near)
            sim.set_counting(counting)
            a = sim.accel()
            if counting:
                np.testing.assert_array_equal(sim.interaction_counts(), counts)
            assert np.abs(a - ref).max() <= bound * big
            sim.close()


@pytest.mark.parametrize("theta", [0.0, 0.15, 0.5, 1.0, 1.5])
@pytest.mark.parametrize("n", [1, 2, 3, 63, 64, 65, 129, 700])
def test_sizes_and_angles(engine, n, theta):
    check(engine, cloud(n, n), theta)


@pytest.mark.parametrize("theta", [-1.0, 1e-200, 1e200])
def test_angles_outside_the_thresholds(engine, theta):
    check(engine, cloud(200, 4), theta)


@pytest.mark.parametrize("kind", ["astro2", "astro"])
@pytest.mark.parametrize("theta,near", [(0.5, 0.0), (1.0, 0.0), (0.5, 1.0), (0.5, 2.0)])
def test_exact_ties(engine, kind, theta, near):
    s = lattice(8)
    if kind == "astro":  # (the quadtree splits by x and y alone)
        s = s[s["z"] == s["z"][0]].copy()
    check(engine, s, theta, near, kind)


def test_fixed_waves_and_short_segments(engine):
    """Waves without a walking body and segments that end inside a wave: each
    member of a batch equals itself alone, bit for bit."""
    states = []
    for i, n in enumerate((1, 5, 64, 130, 300, 2)):
        s = cloud(n, 50 + i)
        if n == 130:
            s["fixed"][:] = True
        if n == 300:
            s["fixed"][::3] = True
        states.append(s)
    kw = dict(theta=0.4, e=0.1, dt=1e-3)
    alone = []
    for s in states:
        sim = P.Sim(engine, s, **kw)
        sim.step(3)
        alone.append(sim.download())
        sim.close()
    sims = [P.Sim(engine, s, **kw) for s in states]
    engine.batch_step(sims, 3)
    for sim, ref in zip(sims, alone):
        np.testing.assert_array_equal(sim.download(), ref)
        sim.close()


@pytest.mark.parametrize("theta", [0.0, -0.0, -1e300, float("-inf"), 5e-324, 1e-121, 2e-121, 1e120,
                                   1.7e120, 1e308, float("inf")])
@pytest.mark.parametrize("kind", ["astro2", "astro"])
def test_angles_around_the_last_thresholds(engine, kind, theta):
    """Squared extent over angle about 2^800 and 2^-800, and past any double:
    an extent of 0.5 to 1 over 1.5e-121 and over 6.7e120."""
    s = cloud(150, 9)
    for f in "xyz":
        s[f] *= 0.75
    check(engine, s, theta, kind=kind)


def test_an_angle_of_zero_costs_no_more_than_a_tiny_one(engine):
    """Both open every cell: the time of the walk, the better of a few passes
    (a division for every test takes 1.6 times as long)."""
    s = cloud(3000, 5)
    best = {}
    engine.set_profiling(True)
    for theta in (1e-9, 0.0, -1.0, 1e-200):
        sim = P.Sim(engine, s, theta=theta, e=0.1)
        for _ in range(6):
            engine.profile_reset()
            sim.accel()
            best[theta] = min(best.get(theta, 1e9), engine.profile()["walk"][0])
        sim.close()
    engine.set_profiling(False)
    print(best)
    assert max(best.values()) <= 1.5 * best[1e-9]
