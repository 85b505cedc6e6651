"""Calls that fail for want of memory leave the engine as it was for the next
one."""
from contextlib import closing

import pytest

import physim_amd as P

pytestmark = pytest.mark.gpu

KW = dict(kind="astro2", theta=1.0, e=0.1, dt=1e-4)


def test_scratch_past_the_device():
    """A batch whose scratch is more than the device has: the call is refused
    as out of memory, and uploads, steps and tree queries go on without it."""
    s = P.cube_and_stars((1 << 20) - 2, seed=3)
    with closing(P.Engine(0, budget=1 << 42)) as eng, closing(P.Engine(0)) as fresh:
        sim = P.Sim(eng, s, **KW)
        sim.accel()  # (leaves extents that the next upload may write to)
        with pytest.raises(P.PgError) as err:
            eng.batch_step([sim] * 120, 1)  # 126 million bodies: 320 GB
        assert err.value.code == 3
        with pytest.raises(P.PgError) as err:
            sim.tree()  # (no build is there any more)
        assert err.value.code == 8
        sim.upload(s)
        sim.step(2)
        ref = P.Sim(fresh, s, **KW)
        ref.step(2)
        assert sim.download().tobytes() == ref.download().tobytes()
        assert sim.stats() == ref.stats()
