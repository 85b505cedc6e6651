"""A server under a tight budget admits what fits with the scratch of all that
it then steps together: every request finishes, some after a wait."""
from contextlib import closing

import numpy as np
import pytest

import physim_amd as P

pytestmark = pytest.mark.gpu


def sphere(n, seed):
    return P.gen_plummer_virial(n, seed=seed, mass=1.0, a=0.1)


@pytest.mark.parametrize("kind,precision", [("simple_astro", "fp64"), ("simple_astro", "mixed"),
                                            ("astro2", "mixed"), ("astro", "fp64")])
def test_requests_past_the_budget_wait(engine, kind, precision):
    kw = dict(kind=kind, precision=precision, theta=0.8, e=0.05, dt=1e-4)
    states = [sphere(n, n) for n in (4099, 3001, 4099, 2500, 4001, 4099, 1200, 4090, 700, 4099)]
    which = {"simple_astro": 0, "astro": 2, "astro2": 3}[kind]
    budget = int(2.7 * P.lib().pg_sim_bytes(4099, which))
    with closing(P.Engine(0, budget=budget)) as eng:
        srv = P.Server(eng)
        ids = [srv.submit(s, 8 + k, **kw) for k, s in enumerate(states)]
        waited = together = 0
        for _ in range(1000):
            active, queued = srv.tick(3)
            waited |= active > 0 and queued > 0
            together |= active > 1
            if active == 0 and queued == 0:
                break
        assert active == 0 and queued == 0 and waited and together
        for k, (rid, s) in enumerate(zip(ids, states)):
            out, info = srv.take(rid, len(s))
            assert info.status == 0
            sim = P.Sim(engine, s, **kw)
            sim.step(8 + k)
            np.testing.assert_array_equal(out, sim.download())
            sim.close()
