"""Launches that only large batches need: a system stepped alone (few node
tiles, its own sort) against the same system stepped beside a filler that
takes the batch past every such line. The tree, the order and the arithmetic
do not depend on it: every bit is compared."""
import numpy as np
import pytest

import physim_amd as P

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def filler():
    return P.gen_plummer_virial(150000, seed=1, mass=1.0, a=0.1)


@pytest.mark.parametrize("kind", ["astro2", "astro"])
@pytest.mark.parametrize("model", ["cube", "plummer"])
@pytest.mark.parametrize("n", [1, 2, 3, 511, 513, 1024, 1025, 2049, 8193, 16384, 16385, 65535,
                               65536, 65537])
def test_alone_equals_beside_a_large_one(engine, filler, kind, model, n):
    if model == "cube" and n > 2:
        s = P.cube_and_stars(n - 2, seed=n)
    else:
        s = P.gen_plummer_virial(n, seed=n, mass=1.0, a=0.1)
    assert len(s) == n
    kw = dict(kind=kind, theta=0.9, e=0.05, dt=1e-4)
    alone, beside, big = (P.Sim(engine, x, **kw) for x in (s, s, filler))
    alone.step(7)
    engine.batch_step([beside, big], 7)
    assert alone.download().tobytes() == beside.download().tobytes()
    a = alone.accel()
    assert a.tobytes() == beside.accel().tobytes()
    for x in (alone, beside, big):
        x.close()


@pytest.mark.parametrize("precision,near", [("fp64", 0.0), ("fp64", 1.5), ("mixed", 1.5)])
@pytest.mark.parametrize("n", [5, 1023, 8192, 8193, 16385, 32768, 32769, 49152, 49153, 98304])
def test_fewer_walking_lanes(engine, filler, precision, near, n):
    """Waves of 4, 8, 16 and 32 walking lanes (alone) against 64 (beside the
    filler), at their lines in both precisions and with a near field."""
    s = P.gen_plummer_virial(n, seed=n, mass=1.0, a=0.1)
    kw = dict(kind="astro2", theta=0.6, e=0.01, dt=1e-4, precision=precision)
    alone, beside, big = (P.Sim(engine, x, **kw) for x in (s, s, filler))
    for x in (alone, beside, big):
        x.set_near_field(near)
        x.set_counting(True)
    alone.step(3)
    engine.batch_step([beside, big], 3)
    assert alone.download().tobytes() == beside.download().tobytes()
    assert alone.interaction_counts().tobytes() == beside.interaction_counts().tobytes()
    for x in (alone, beside, big):
        x.close()


@pytest.mark.parametrize("pairs", [0, 20, 30, 36, 42, 60])
def test_tiles_around_the_node_list(engine, pairs):
    """One node tile of a quadtree whose internal nodes go from 0.7 to 1.2 per
    body: up to 992 are built one per thread, more body by body."""
    from oracle import oracle as O

    rng = np.random.default_rng(pairs)
    s = np.zeros(1024, P.ENTITY)
    for f in "xyz":
        s[f] = rng.uniform(-1.0, 1.0, len(s))
    for f in "xy":  # (bodies near another: a chain of cells each)
        s[f][:pairs] = s[f][512:512 + pairs] + rng.uniform(1e-4, 2e-4, pairs)
    s["mass"] = rng.uniform(0.5, 1.5, len(s))
    ref, _, fault = O.bh_transform(s, 0.7, 0.1, 2)
    assert fault == 0
    a = P.Sim(engine, s, kind="astro", theta=0.7, e=0.1, precision="fp64").accel()
    r = np.linalg.norm(a - ref, axis=1) / np.linalg.norm(ref, axis=1)
    assert np.quantile(r, 0.99) <= 1e-11 and r.max() <= 1e-8


@pytest.mark.parametrize("pairs,run", [(1, 2), (10, 2), (339, 2), (340, 2), (341, 2), (700, 2),
                                       (40, 3), (16, 40), (4, 64), (3, 65), (2, 256)])
def test_tied_first_words(engine, pairs, run):
    """`pairs` runs of `run` bodies in one cell of level 21 each, beside single
    ones, in one bucket: up to 680 tied bodies are ordered from LDS, more (and
    runs past a slot's 64 keys) run by run. First and later passes against the
    radix sort's, which orders every run by one thread: the same bits."""
    rng = np.random.default_rng(pairs * 1000 + run)
    n = pairs * run + 50
    s = np.zeros(n, P.ENTITY)
    cells = rng.choice(1 << 18, pairs, replace=False)
    for k, f in enumerate("xyz"):
        s[f][:pairs * run] = np.repeat(((cells >> (6 * k)) & 63) / 64.0, run) + 2e-7 \
            + rng.uniform(0.0, 5e-7, pairs * run)
        s[f][pairs * run:] = rng.uniform(-1.0, 0.0, 50)
    s["x"][-1] = -1.0  # the extent: cells of level 21 are 2^-20 wide
    s["mass"] = rng.uniform(0.5, 1.5, n)
    kw = dict(kind="astro2", theta=0.7, e=0.1, precision="fp64")
    radix = P.Engine(0)
    radix.set_sort(max_buckets=0)
    other = P.Sim(radix, s, **kw)
    sim = P.Sim(engine, s, **kw)
    for _ in range(3):
        assert sim.accel().tobytes() == other.accel().tobytes()
    assert sim.stats() == other.stats()
    sim.close()
    radix.close()


@pytest.mark.parametrize("n", [700, 1900, 3000, 9000, 16384, 16385])
def test_keys_far_from_the_last_splitters(engine, n):
    """A state whose keys all fall in one or two of the buckets that the
    previous state's keys made (up to 2,048 keys listed, more written out for
    the other sorts), against a fresh engine."""
    rng = np.random.default_rng(n)
    s = np.zeros(n, P.ENTITY)
    for f in "xyz":
        s[f] = rng.uniform(-1.0, 1.0, n)
    s["mass"] = 1.0 / n
    kw = dict(kind="astro2", theta=0.7, e=0.1)
    sim = P.Sim(engine, s, **kw)
    sim.accel()
    for f in "xyz":
        s[f][1:] = 0.9 + s[f][1:] * 1e-3
    s["x"][0] = -1.0
    sim.upload(s)
    fresh = P.Engine(0)
    ref = P.Sim(fresh, s, **kw)
    for _ in range(2):
        assert sim.accel().tobytes() == ref.accel().tobytes()
    sim.close()
    fresh.close()
