"""GPU: rounding of the fast build's kicks against extended precision, by the
form of the field. A magnet of 10 slices kicks a particle 30 times; each kick
rounds px and py once, so the error of a particle is a random walk of 30 steps
of rms 0.29 units in the last place: 1.6 units. A product that is rounded alike at
every kick adds up instead, to 30 x 0.25 units on average. Bound: 2.4 units
(half as much again for the coordinates that the kick is computed from)."""

import numpy as np
import pytest

from at_amd import engine
from at_amd.lattice import Dipole, Lattice, Octupole, Particle, Sextupole

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(np.finfo(np.longdouble).eps > 2e-19,
                                 reason="no extended precision on this machine")]

N, SLICES = 20000, 10
# the engine's Forest-Ruth coefficients, with their roundings
CBRT2 = 1.25992104989487316477
DRIFT = (1.0 / (2.0 * (2.0 - CBRT2)), 0.5 - (1.0 / (2.0 * (2.0 - CBRT2))))
KICK = (1.0 / (2.0 - CBRT2), 1.0 - 2.0 / (2.0 - CBRT2))


def _exact(m, beam):
    """The magnet's slices in extended precision, from the same double constants."""
    ld = np.longdouble
    x, px, y, py, dp, ct = beam.astype(ld)
    a, b = [ld(v) for v in m.PolynomA], [ld(v) for v in m.PolynomB]
    step = m.Length / m.NumIntSteps
    irho = ld(getattr(m, "BendingAngle", 0.0) / m.Length)
    d1, d2, k1, k2 = (ld(step * v) for v in DRIFT + KICK)
    p = 1 / (1 + dp)
    for _ in range(m.NumIntSteps):
        for d, k in ((d1, k1), (d2, k2), (d2, k1), (d1, None)):
            x, y = x + d * p * px, y + d * p * py
            ct = ct + d * p * p * (px * px + py * py) / 2
            if k is None:
                continue
            re, im = b[-1], a[-1]
            for i in range(len(a) - 2, -1, -1):
                re, im = re * x - im * y + b[i], im * x + re * y + a[i]
            px, py = px - k * (re - (dp - x * irho) * irho), py + k * im
            ct = ct + k * irho * x
    return np.array([x, px, y, py, dp, ct])


def _pass(m, beam):
    ring = Lattice([m], energy=3.0e9, particle=Particle("electron"), name="one")
    dl = engine.DeviceLattice(ring)
    try:
        got = beam.copy(order="F")
        dl.track(got, 1, None, energy=ring.energy, rest_energy=ring.particle.rest_energy)
    finally:
        dl.close()
    return got


def _beam(scale):
    return np.asfortranarray(np.random.default_rng(21).uniform(-1.0, 1.0, (6, N))
                             * np.array(scale)[:, None])


def _rms_units(got, exact):
    units = (got - exact).astype(float) / np.spacing(np.abs(got))
    units = units[np.abs(got) > 2e-5]  # a coordinate that passes zero keeps larger roundings
    return np.sqrt(np.mean(units * units))


@pytest.mark.parametrize("s", [0.55, 0.8, 1.1, 1.45])
def test_sextupole_with_steerer(s):
    m = Sextupole("S", 0.2, 120.0 * s, PolynomB=[1e-5 * s, 0.0, 120.0 * s],
                  PolynomA=[-2e-5 * s, 0.0, 0.0], NumIntSteps=SLICES)
    beam = _beam([1e-3, 1e-4, 1e-3, 1e-4, 1e-3, 1e-3])
    exact, got = _exact(m, beam), _pass(m, beam)
    for k in (1, 3):
        assert _rms_units(got[k], exact[k]) < 2.4


@pytest.mark.parametrize("s", [0.55, 0.8, 1.1, 1.25])
def test_octupole_strength(s):
    """The part of the error that is proportional to the kick, as a relative error of the
    strength. The remainder of the product is added once, at the first kick: a coordinate that
    changes by less than 0.4 leaves 0.4 x 1.1e-16, and the roundings of 20,000 particles
    2e-17 (5 sigma). Without the remainder: up to 1.1e-16 and the sum of two of them."""
    m = Octupole("O", 0.05, [0, 0, 0, 0], [0, 0, 0, 60000.0 * s], NumIntSteps=SLICES)
    beam = _beam([8e-3, 1e-5, 8e-3, 1e-5, 1e-3, 1e-3])
    exact, got = _exact(m, beam), _pass(m, beam)
    for k in (1, 3):
        kick = (exact[k] - beam[k]).astype(float)
        err = (got[k] - exact[k]).astype(float)
        assert abs(np.sum(err * kick) / np.sum(kick * kick)) < np.finfo(float).eps / 3


@pytest.mark.parametrize("s", [0.55, 0.8, 1.1, 1.45])
def test_bend_with_gradient(s):
    """One rounding per kick: 1.58 units, and a hundredth of that for 20,000 particles (the
    curvature and the gradient kicked one after the other make two, the second on a smaller
    coordinate: 1.8)."""
    m = Dipole("B", 1.0, 0.02 * s, -0.6 * s, NumIntSteps=SLICES)
    beam = _beam([8e-3, 1e-4, 4e-3, 1e-4, 1e-3, 1e-3])
    exact, got = _exact(m, beam), _pass(m, beam)
    assert _rms_units(got[1], exact[1]) < 1.65
