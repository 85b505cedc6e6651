"""States and results on their way through the engine's pinned memory, at the
sizes where the path changes: a state up to 256 KiB is unpacked in place
(3,276 records of 80 bytes), accelerations up to that size come with the status
(10,922 bodies), larger ones move in chunks of 3 MiB (39,321 records, 131,072
bodies), two of them in use. Copies are exact, so every comparison is."""
import numpy as np
import pytest

import physim_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 255, 257, 3276, 3277, 39321, 39322, 78643, 78644, 200001])
def test_state_round_trip(engine, n):
    rng = np.random.default_rng(n)
    s = np.frombuffer(rng.bytes(n * P.ENTITY.itemsize), P.ENTITY).copy()
    for f in ("x", "y", "z", "vx", "vy", "vz", "radius", "mass"):
        s[f] = rng.uniform(-1.0, 1.0, n)
    sim = P.Sim(engine, s, kind="astro2")
    assert sim.download().tobytes() == s.tobytes()
    back = s[::-1].copy()  # (a contiguous array is uploaded as it is, padding and all)
    sim.upload(back)
    assert sim.download().tobytes() == back.tobytes()
    sim.close()


@pytest.mark.parametrize("n", [1, 2, 3277, 10922, 10923, 131072, 131073, 262146])
def test_transform_adds_the_pass(engine, n):
    rng = np.random.default_rng(n)
    s = np.zeros(n, P.ENTITY)
    for f in "xyz":
        s[f] = rng.uniform(-1.0, 1.0, n)
    s["mass"] = 1.0 / n
    before = rng.uniform(-1.0, 1.0, (n, 3))
    acc = np.zeros(n, P.ACCEL)
    for k, f in enumerate("xyz"):
        acc[f] = before[:, k]
    sim = P.Sim(engine, s, kind="astro2", theta=1.5, e=0.1)
    a = sim.accel()
    sim.close()
    got = engine.transform(s, kind="astro2", theta=1.5, e=0.1, acc=acc)
    assert got.view(np.float64).reshape(-1, 3).tobytes() == (before + a).tobytes()


def test_device_tables_follow_the_batch():
    """Steps of one simulation, another, both and either again (the tables kept,
    with their parities changed over, or written anew), against each simulation
    stepped on an engine of its own."""
    states = [P.gen_plummer_virial(n, seed=n, mass=1.0, a=0.1) for n in (3000, 5001)]
    kw = dict(kind="astro2", theta=0.7, e=0.01, dt=1e-4)
    both = P.Engine(0)
    sims = [P.Sim(both, s, **kw) for s in states]
    alone = [P.Engine(0) for _ in states]
    refs = [P.Sim(e, s, **kw) for e, s in zip(alone, states)]
    for op, steps in ((0, 1), (0, 1), (0, 2), (1, 1), (0, 1), (2, 3), (2, 1), (2, 4), (1, 3),
                      (1, 6), (2, 5), (0, 7)):
        if op == 2:
            both.batch_step(sims, steps)
        else:
            sims[op].step(steps)
        for k in (0, 1):
            if op in (k, 2):
                refs[k].step(steps)
    sims[0].set_params(kind="simple_astro", theta=0.7, e=0.01, dt=1e-4)
    refs[0].set_params(kind="simple_astro", theta=0.7, e=0.01, dt=1e-4)
    sims[0].step(2)
    refs[0].step(2)
    for a, b in zip(sims, refs):
        assert a.download().tobytes() == b.download().tobytes()
    for e in [both] + alone:
        e.close()


@pytest.mark.parametrize("integrator", ["euler", "rk4"])
def test_failed_pass_leaves_the_state(engine, integrator):
    """A step whose acceleration pass fails on the device reports it and
    changes nothing, now and when it is asked for again."""
    s = P.cube_and_stars(2000, seed=6)
    s["z"][11] = np.inf
    sim = P.Sim(engine, s, kind="astro2", theta=1.0, e=0.5)
    sim.set_integrator(integrator)
    for _ in range(2):
        with pytest.raises(P.PgError) as ei:
            sim.step(2)
        assert ei.value.code == 7
        assert sim.download().tobytes() == s.tobytes()
    sim.close()


@pytest.mark.parametrize("n", [1, 255, 257, 4095, 4097, 20000])
@pytest.mark.parametrize("kind", ["astro2", "astro"])
def test_extent_of_uploads_and_stages(engine, kind, n):
    """The extent left by an upload after a force-only pass, and by each euler
    and rk4 stage, against passes of a fresh engine, which reduce it from the
    positions: states that grow and shrink, the largest coordinate in any block
    and on any axis, non-finite ones. Also through a change to the direct sum
    and back, whose steps leave no extent."""
    rng = np.random.default_rng(n)
    base = np.zeros(n, P.ENTITY)
    for f in ("x", "y", "z", "vx", "vy", "vz"):
        base[f] = rng.uniform(-1.0, 1.0, n)
    base["mass"] = 1.0 / n
    kw = dict(kind=kind, theta=0.7, e=0.1)
    fresh = P.Engine(0)
    for k in range(6):
        s = base.copy()
        s["xyz"[k % 3]][rng.integers(n)] = (-1.0) ** k * 10.0 ** (2 - k)
        a = engine.transform(s, **kw)
        ref = P.Sim(fresh, s, **kw)
        assert a.view(np.float64).reshape(-1, 3).tobytes() == ref.accel().tobytes()
        ref.close()
        bad = s.copy()
        bad["xyz"[k % 3]][rng.integers(n)] = (np.inf, -np.inf, np.nan)[k // 2]
        with pytest.raises(P.PgError) as ei:
            engine.transform(bad, **kw)
        assert ei.value.code == 7
    for integrator in ("euler", "rk4"):
        sim = P.Sim(engine, base, dt=0.1, **kw)
        sim.set_integrator(integrator)
        for _ in range(3):
            sim.step(1)
            now = P.Sim(fresh, sim.download(), **kw)
            assert sim.accel().tobytes() == now.accel().tobytes()
            now.close()
        sim.set_params(kind="simple_astro", theta=0.7, e=0.1, dt=0.5)
        sim.step(2)
        sim.set_params(dt=0.1, **kw)
        now = P.Sim(fresh, sim.download(), **kw)
        assert sim.accel().tobytes() == now.accel().tobytes()
        now.close()
        sim.close()
    fresh.close()
