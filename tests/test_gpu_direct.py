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
