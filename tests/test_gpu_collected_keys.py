"""The sort whose blocks collect their own keys (batches of up to 16,384
bodies), where some of its buckets are sorted in global memory while other
blocks still read the unsorted keys: the radix sort's order and tree, bit for
bit."""
import threading

import numpy as np
import pytest

import physim_amd as P

pytestmark = pytest.mark.gpu

KW = dict(kind="astro2", theta=0.7, e=0.1)


def cube(n, seed):
    rng = np.random.default_rng(seed)
    s = np.zeros(n, P.ENTITY)
    for f in "xyz":
        s[f] = rng.uniform(-1.0, 1.0, n)
    s["x"][0] = -1.0  # (the extent stays as it is)
    s["mass"] = rng.uniform(0.5, 1.5, n) / n
    return s


def against_radix(states, cap, engine=None):
    """Passes over `states` with buckets above `cap` keys sorted in global
    memory, against the radix sort's."""
    eng = engine or P.Engine(0)
    eng.set_sort(bucket_cap=cap)
    radix = P.Engine(0)
    radix.set_sort(max_buckets=0)
    sim, ref = P.Sim(eng, states[0], **KW), P.Sim(radix, states[0], **KW)
    same = []
    for s in states:
        sim.upload(s)
        ref.upload(s)
        same.append(sim.accel().tobytes() == ref.accel().tobytes() and sim.stats() == ref.stats())
    sim.close()
    ref.close()
    radix.close()
    if engine is None:
        eng.close()
    return same


@pytest.mark.parametrize("cap", [0, 100, 384, 4096])
@pytest.mark.parametrize("n", [2, 1025, 5001, 16384])
def test_buckets_past_the_cap(n, cap):
    assert all(against_radix([cube(n, k) for k in range(4)], cap))


@pytest.mark.parametrize("crowd", [2047, 2049, 4095, 4097, 9000])
def test_one_bucket_past_the_cap(crowd):
    """One bucket of the previous keys takes `crowd` bodies (4,096 fit LDS),
    the others stay as they were and are collected beside it."""
    a = cube(16384, 1)
    b = a.copy()
    for f in "xyz":
        b[f][1:crowd + 1] = 0.9 + b[f][1:crowd + 1] * 1e-3
    assert all(against_radix([a, b, a, b, b], 4096))


def test_buckets_past_the_cap_on_a_busy_gpu():
    """Four engines at once, so that blocks of one launch start far apart."""
    got = [None] * 4

    def work(k):
        got[k] = against_radix([cube(16384 - k, 10 * k + i) for i in range(6)], 200)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(g and all(g) for g in got)


@pytest.mark.parametrize("cap", [0, 100, 4096])
@pytest.mark.parametrize("n,run", [(900, 3), (3000, 2), (3000, 5), (9000, 30), (9000, 70),
                                   (16384, 4), (16385, 4)])
def test_runs_of_equal_keys_at_bucket_ends(n, run, cap):
    """Bodies in runs of one cell of level 21 each, so that buckets begin and
    end with a run; between passes some leave a run for one before or after
    it, so that the previous pass's keys just past a bucket are its own first
    or last key."""
    rng = np.random.default_rng(n + run)
    s = np.zeros(n, P.ENTITY)
    cells = rng.choice(1 << 18, n // run + 1, replace=False)

    def put(i, c):
        for k, f in enumerate("xyz"):
            s[f][i] = ((c >> (6 * k)) & 63) / 64.0 + 2e-7 + rng.uniform(0.0, 5e-7, len(i))

    s["mass"] = rng.uniform(0.5, 1.5, n) / n
    put(np.arange(n), np.repeat(cells, run)[:n])
    s["x"][0] = -1.0  # (the extent: cells of level 21 are 2^-20 wide)
    states = [s.copy()]
    for _ in range(5):
        some = rng.choice(np.arange(1, n), n // 8, replace=False)
        put(some, rng.choice(cells, len(some)))
        states.append(s.copy())
    assert all(against_radix(states, cap))
