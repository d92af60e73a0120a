"""GPU: coordinates that overflow inside a magnet, and infinite ones that enter
it, against the oracle, by the transforms that the magnet has: shifts only, a
roll at one end only, all, none. A transform that is missing leaves a coordinate
as it is (no zero times an infinity), one that is there spreads NaN through the
zeros of its matrix. Strict build: bit for bit. Fast build: its FMAs have no
product that overflows by itself, so that an infinity of its may be a NaN of the
oracle's (inf - inf); what is not finite is compared, bit for bit, with the same
magnet run by the general form of the map (which a shift of delta selects, by far
less than its last place), finite values to 1e-8 (each of the 6 kicks raises a coordinate to at
most its third power, so 3^6 roundings of 2e-16, and a thousandfold for
differences of coordinates that nearly cancel)."""

import numpy as np
import pytest

from at_amd import engine
from at_amd.lattice import Drift, Lattice, Octupole, Particle, Quadrupole, Sextupole
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

RAD = "StrMPoleSymplectic4RadPass"
MOVES = ["none", "shift", "r1", "r2", "all"]


def _move(m, how):
    c, s = np.cos(1e-3), np.sin(1e-3)
    roll = np.eye(6)
    roll[0, 0] = roll[1, 1] = roll[2, 2] = roll[3, 3] = c
    roll[0, 2] = roll[1, 3] = s
    roll[2, 0] = roll[3, 1] = -s
    if how in ("shift", "all"):
        m.T1 = np.array([1e-4, 0.0, -2e-4, 0.0, 0.0, 0.0])
        m.T2 = -m.T1
    if how in ("r1", "all"):
        m.R1 = roll
    if how in ("r2", "all"):
        m.R2 = roll.T.copy()
    return m


def _magnet(kind, slices):
    if kind == "sext":
        m = Sextupole("S", 0.3, 2000.0)
    elif kind == "steerer":
        m = Sextupole("S", 0.3, 2000.0, PolynomB=[1e-4, 0.0, 2000.0], PolynomA=[-2e-4, 0.0, 0.0])
    elif kind == "oct":
        m = Octupole("O", 0.3, [0, 0, 0, 0], [0, 0, 0, 3000.0])
    else:
        m = Quadrupole("Q", 0.4, 20.0, PassMethod=RAD)  # radiates all its energy
    m.NumIntSteps = slices
    return m


def _ring(m):
    # the drift before it is the call's first element, so the magnet runs by its record
    return Lattice([Drift("D", 0.1), Drift("D", 0.1), m, Drift("D", 0.1)], energy=4.0e10,
                   particle=Particle("electron"), name="overflow")


def _track(ring, beam, strict, losses=True):
    r = beam.copy(order="F")
    dl = engine.DeviceLattice(ring)
    try:
        out = dl.track(r, 1, None, energy=ring.energy, rest_energy=ring.particle.rest_energy,
                       losses=losses, strict=strict)
    finally:
        dl.close()
    return r, out[1] if losses else None


@pytest.mark.parametrize("how", MOVES)
@pytest.mark.parametrize("kind,slices", [("sext", 10), ("steerer", 10), ("oct", 2), ("quad", 10)])
def test_loss_coordinates(kind, slices, how):
    n = 2000
    rng = np.random.default_rng(11)
    beam = np.asfortranarray(1e-3 * rng.standard_normal((6, n)))
    beam[0] = rng.uniform(0.2, 0.99, n)
    beam[2] = rng.uniform(0.0, 0.9, n) * rng.integers(0, 2, n)
    ring = _ring(_move(_magnet(kind, slices), how))
    ref = beam.copy(order="F")
    _, want = po.atpass(ring, ref, 1, losses=True)
    wild = ~np.isfinite(want["coord"])
    assert wild.any() and (want["elem"][wild.any(axis=0)] == 2).all()
    got, have = _track(ring, beam, True)
    for k in ("islost", "turn", "elem", "coord"):
        np.testing.assert_array_equal(have[k], want[k], err_msg=k)
    np.testing.assert_array_equal(got, ref)
    if slices > 2:
        return
    got, have = _track(ring, beam, False)
    ring[2].T1 = getattr(ring[2], "T1", np.zeros(6)) + np.array([0, 0, 0, 0, 1e-300, 0])
    ref, want = _track(ring, beam, False)
    for k in ("islost", "turn", "elem"):
        np.testing.assert_array_equal(have[k], want[k], err_msg=k)
    wild = ~np.isfinite(want["coord"]).all(axis=0) | ~np.isfinite(have["coord"]).all(axis=0)
    assert wild.any()
    np.testing.assert_array_equal(have["coord"][:, wild], want["coord"][:, wild])
    np.testing.assert_allclose(have["coord"], want["coord"], rtol=1e-8, atol=1e-8)
    np.testing.assert_allclose(got, ref, rtol=1e-8, atol=1e-8)


@pytest.mark.parametrize("kind,slices", [("sext", 2), ("steerer", 2), ("oct", 1)])
def test_finite_loss_coordinates(kind, slices):
    """Particles that a strong multipole throws far out, but not to infinity: each kick raises the
    relative error to its power at most, as above, in the fast build as well."""
    n = 2000
    rng = np.random.default_rng(14)
    beam = np.asfortranarray(1e-3 * rng.standard_normal((6, n)))
    beam[0], beam[2] = rng.uniform(0.2, 0.99, n), rng.uniform(0.0, 0.9, n)
    ring = _ring(_magnet(kind, slices))
    ref = beam.copy(order="F")
    _, want = po.atpass(ring, ref, 1, losses=True)
    assert np.abs(want["coord"][0]).max() > 1e20 and np.isfinite(want["coord"]).all()
    for strict in (True, False):
        got, have = _track(ring, beam, strict)
        for k in ("islost", "turn", "elem"):
            np.testing.assert_array_equal(have[k], want[k], err_msg=k)
        np.testing.assert_allclose(have["coord"], want["coord"], rtol=0 if strict else 1e-8, atol=0)


@pytest.mark.parametrize("how", MOVES)
@pytest.mark.parametrize("kind,slices", [("sext", 2), ("oct", 2), ("quad", 2)])
def test_infinite_input_without_loss_records(kind, slices, how):
    """Without loss records an infinite x is not replaced: elements go on with it."""
    beam = np.asfortranarray(1e-3 * np.random.default_rng(12).standard_normal((6, 80)))
    beam[0, 10], beam[0, 11] = np.inf, -np.inf
    beam[:, 12] = [np.inf, 0.0, 0.0, 0.0, 0.0, 0.0]
    beam[0, 13], beam[2, 13] = np.inf, np.inf
    ring = _ring(_move(_magnet(kind, slices), how))
    ref = beam.copy(order="F")
    po.atpass(ring, ref, 1)
    got, _ = _track(ring, beam, True, losses=False)
    np.testing.assert_array_equal(got, ref)
    got, _ = _track(ring, beam, False, losses=False)
    np.testing.assert_allclose(got, ref, rtol=1e-12, atol=1e-12)


@pytest.mark.parametrize("how", MOVES)
def test_signs_of_zero(how):
    """Strict build: a particle at (signed) zeros passes a magnet without kicks as in the oracle."""
    beam = np.zeros((6, 64), order="F")
    beam[np.random.default_rng(13).integers(0, 2, (6, 64)) == 1] = -0.0
    m = _move(Quadrupole("Q", 0.4, 0.0), how)
    for t in ("T1", "T2"):
        if how == "all":
            setattr(m, t, np.array([0.0, -0.0, -0.0, 0.0, 0.0, 0.0]))
    ring = _ring(m)
    ref = beam.copy(order="F")
    po.atpass(ring, ref, 1)
    got, _ = _track(ring, beam, True, losses=False)
    np.testing.assert_array_equal(np.signbit(got), np.signbit(ref))
