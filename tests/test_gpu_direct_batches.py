"""Direct sums whose partial sums do not fit one launch: formed a run of target
tiles at a time, with the bits that every simulation has alone."""
from contextlib import closing

import numpy as np
import pytest

import physim_amd as P

pytestmark = pytest.mark.gpu


def bodies(n, seed):
    rng = np.random.default_rng(seed)
    s = np.zeros(n, P.ENTITY)
    for f in "xyz":
        s[f] = rng.uniform(-1.0, 1.0, n)
        s["v" + f] = rng.normal(size=n)
    s["mass"] = rng.uniform(0.5, 1.5, n) / n
    s["fixed"][::5] = True
    return s


def alone(engine, s, steps, **kw):
    sim = P.Sim(engine, s, **kw)
    sim.step(steps)
    out = sim.download()
    acc = sim.accel()
    sim.close()
    return out.tobytes(), acc.tobytes()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_many_members_in_bounded_scratch(engine, precision):
    """48 members whose partial sums are 600 MB together (FP64): the scratch
    holds 64 MB of them beside its share of each body, and every member has
    the bits it has alone, stepped and replayed from a graph."""
    kw = dict(kind="simple_astro", precision=precision, e=0.1, dt=1e-4)
    sizes = [(8195, 4097, 1, 300, 18900, 2048)[k % 6] for k in range(48)]
    states = [bodies(n, k) for k, n in enumerate(sizes)]
    with closing(P.Engine(0)) as eng:
        sims = [P.Sim(eng, s, **kw) for s in states]
        before = eng.memory()[0]
        eng.batch_step(sims, 7)
        scratch = eng.memory()[0] - before
        # (72 bytes of node arrays for 64 of partial sums; 200 bytes a body)
        assert scratch <= (64 << 20) * 9 // 8 + 200 * sum(sizes) + (1 << 20)
        for k in (0, 1, 2, 3, 4, 5, 24, 46, 47):
            assert sims[k].download().tobytes() == alone(engine, states[k], 7, **kw)[0]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [1025, 4097, 8195, 18689, 18900, 65537])
def test_one_member_in_a_tight_budget(engine, n, precision):
    """What pg_sim_bytes names is enough for a pass (and 400 KB for the
    engine's own), and its partial sums then take several rounds."""
    kw = dict(kind="simple_astro", precision=precision, e=0.1, dt=1e-4)
    s = bodies(n, n)
    ref = alone(engine, s, 6, **kw)
    need = P.lib().pg_sim_bytes(n, 0)
    for budget in (need + 400_000, need * 3 // 2, need * 4):
        with closing(P.Engine(0, budget=budget)) as eng:
            assert alone(eng, s, 6, **kw) == ref
            assert eng.memory()[0] <= budget


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_batch_in_a_tight_budget(engine, precision):
    kw = dict(kind="simple_astro", precision=precision, e=0.1, dt=1e-4)
    states = [bodies(n, n) for n in (700, 4097, 255, 8195, 2049)]
    budget = sum(P.lib().pg_sim_bytes(len(s), 0) for s in states)
    with closing(P.Engine(0, budget=budget)) as eng:
        sims = [P.Sim(eng, s, **kw) for s in states]
        eng.batch_step(sims, 5)
        for sim, s in zip(sims, states):
            assert sim.download().tobytes() == alone(engine, s, 5, **kw)[0]


@pytest.mark.parametrize("n", [18688, 18689, 18893, 18894])
def test_allocation_free_in_two_rounds(engine, n):
    """Its node array holds 5,461 lines of partial sums: 73 x 73 tiles, not 74 x 74."""
    s = bodies(n, n)
    kw = dict(kind="simple_astro", precision="mixed", e=0.1)
    for _ in range(2):
        assert engine.transform_noalloc(s, **kw).tobytes() == engine.transform(s, **kw).tobytes()
