"""A tuning's bucket size is used as it is named; the default follows the
batch's size. A batch past lds_buckets buckets takes its splitters from a
kernel of their own in every step, so the number of buckets shows there."""
from contextlib import closing

import pytest

import physim_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,bucket_keys,buckets", [
    (36000, 1664, 94), (36000, 384, 94), (36000, 383, 94), (36000, 2048, 18), (36000, 1280, 29),
    (36000, 256, 141), (131072, 1664, 342), (131073, 1664, 129), (131072, 1280, 103),
    (400000, 1664, 391), (400000, 1280, 313), (400000, 2048, 196), (600000, 1664, 361)])
def test_bucket_keys_in_use(n, bucket_keys, buckets):
    with closing(P.Engine(0)) as eng:
        sim = P.Sim(eng, P.cube_and_stars(n - 2, seed=1), kind="astro2", theta=1.5, e=0.1, dt=1e-6)
        eng.set_profiling(True)
        for most in (buckets, buckets - 1):
            eng.set_tuning(bucket_keys=bucket_keys, lds_buckets=most)
            assert eng.tuning()["bucket_keys"] == bucket_keys
            sim.step(2)
            eng.profile_reset()
            sim.step(4)
            assert eng.profile().get("splitters", (0.0, 0))[1] == (0 if most == buckets else 4)
