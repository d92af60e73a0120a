"""GPU: the thick multipoles that the tracking kernel runs by their records, of all
orders that have one, with each of the maps around them, and drifts, markers and
correctors with apertures, against the oracle. Strict build: bit for bit; fast
build: a magnet's few hundred roundings of coordinates below 1 stay below 1e-12, and
the loss records are the same. And the change of the loop over the records in the
middle of a turn: a particle outside the ranges of the kicks' series changes no bit
of the others of its wave."""

import numpy as np
import pytest

from at_amd import engine
from at_amd.lattice import (Aperture, Corrector, Dipole, Drift, Lattice, Marker, Multipole, Particle,
                            Quadrupole, RFCavity, Sextupole, ThinMultipole)
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

A = [4e-4, -0.2, 2.0, 30.0]
B = [3e-4, 0.9, -8.0, 200.0]
FIELDS = ["none", "lead", "first", "dipole", "all"]
AROUND = ["none", "rect", "ellipse", "scale", "shift", "roll", "matrix", "fringe", "edges", "both"]


def _rot(psi):
    c, s = np.cos(psi), np.sin(psi)
    r = np.eye(6)
    r[0, 0] = r[1, 1] = r[2, 2] = r[3, 3] = c
    r[0, 2] = r[1, 3] = s
    r[2, 0] = r[3, 1] = -s
    return r


def _field(field, order):
    a, b = np.zeros(max(order, 1) + 1), np.zeros(max(order, 1) + 1)
    if field == "lead":
        b[order] = B[order]
    elif field == "first":  # as of a lower order
        b[min(order, 1)] = B[min(order, 1)]
    elif field == "dipole":
        a[0], b[0], b[order] = A[0], B[0], B[order]
    elif field == "all":
        a[:order + 1], b[:order + 1] = A[:order + 1], B[:order + 1]
    return a, b


def _around(m, how, bend):
    if how in ("rect", "both"):
        m.RApertures = np.array([-2.5e-3, 2e-3, -2e-3, 1.5e-3])
    if how in ("ellipse", "both"):
        m.EApertures = np.array([3e-3, 2.5e-3])
    if how in ("scale", "both"):
        m.FieldScaling = 1.003
    if how in ("shift", "both"):
        m.T1, m.T2 = np.array([1e-4, 0, -2e-4, 1e-5, 0, 0]), np.array([-1e-4, 0, 2e-4, 0, 0, 0])
    if how in ("roll", "both"):
        m.R1, m.R2 = _rot(1e-3), _rot(-2e-3)
    if how == "matrix":
        r = _rot(1e-3)
        r[0, 4], r[5, 1] = 1e-4, -1e-4
        m.R1, m.R2 = r, np.linalg.inv(r)
        m.T1, m.T2 = np.array([1e-4, 0, 0, 0, 0, 1e-4]), np.array([0, 0, 0, 0, 1e-4, 0])
    if how in ("fringe", "both"):
        m.FringeQuadEntrance, m.FringeQuadExit = 1, 1
    if how == "edges" and bend:
        m.FringeBendEntrance, m.FringeBendExit = 2, 2
        m.FullGap, m.FringeInt1, m.FringeInt2 = 0.02, 0.5, 0.5
    return m


def _beam(n=200):
    r = np.asfortranarray(np.random.default_rng(7).standard_normal((6, n))
                          * np.array([1e-3, 2e-4, 1e-3, 2e-4, 1e-3, 1e-3])[:, None])
    r[1, 40:43] = [0.02, -0.03, 0.011]  # wide angles, in one wave
    return r


def _check(ring, beam, turns, refs=None):
    rest = ring.particle.rest_energy
    ref = beam.copy(order="F")
    out, want = po.atpass(ring, ref, turns, refpts=refs, losses=True)
    dl = engine.DeviceLattice(ring)
    try:
        for strict in (True, False):
            got = beam.copy(order="F")
            copies, have = dl.track(got, turns, refs, energy=ring.energy, rest_energy=rest,
                                    losses=True, strict=strict)
            for k in ("islost", "turn", "elem"):
                np.testing.assert_array_equal(have[k], want[k], err_msg=f"{strict} {k}")
            for x, y in ((got, ref), (have["coord"], want["coord"]), (copies, out)):
                if y is None:
                    continue
                if strict:
                    np.testing.assert_array_equal(x, y)
                else:
                    np.testing.assert_allclose(x, y, rtol=1e-12, atol=1e-12)
    finally:
        dl.close()
    return want


@pytest.mark.parametrize("order", [0, 1, 2, 3])
@pytest.mark.parametrize("rad", [False, True], ids=["plain", "rad"])
@pytest.mark.parametrize("bend", [False, True], ids=["straight", "bend"])
def test_kinds(bend, rad, order):
    method = ("Bnd" if bend else "Str") + "MPoleSymplectic4" + ("Rad" if rad else "") + "Pass"
    lost = 0
    for how in AROUND:
        elems = [Drift("D", 0.05)]
        for i, field in enumerate(FIELDS):
            a, b = _field(field, order)
            if bend:
                m = Dipole("B", 0.4, 0.02, 0.0, EntranceAngle=0.01, ExitAngle=0.012)
            else:
                m = Multipole("M", 0.3, a, b)
            m.PassMethod, m.PolynomA, m.PolynomB, m.MaxOrder = method, a, b, order
            m.NumIntSteps = 1 + 2 * i
            elems += [Drift("D", 0.05), _around(m, how, bend)]
        for energy in (3.0e9, 4.0e10):  # radiated fractions per kick below and above 2e-6
            ring = Lattice(elems + [Drift("D", 0.05)], energy=energy, particle=Particle("electron"),
                           name=how)
            want = _check(ring, _beam(), 1)
            _check(ring, _beam(70), 2, np.arange(len(ring) + 1, dtype=np.uint32))
            lost += int(want["islost"].sum())
            assert want["islost"].sum() < 150
    assert lost > 0


def test_apertures_on_other_elements():
    rect = {"RApertures": np.array([-2e-3, 2e-3, -1.5e-3, 1.5e-3])}
    ellipse = {"EApertures": np.array([2.5e-3, 2e-3])}
    both = {**rect, **ellipse}
    elems = [Drift("D", 0.05)]
    for ap in (rect, ellipse, both):
        elems += [Marker("M", **ap), Drift("D", 0.1), Drift("D", 0.1, **ap), Marker("M"),
                  Corrector("C", 0.0, [1e-4, -2e-4], **ap), Corrector("C", 0.1, [1e-4, 2e-4], **ap),
                  ThinMultipole("T", [0, 0, 0], [0, 0, 3.0], **ap), Drift("D", 0.1),
                  ThinMultipole("T", [0, 0, 0, 0], [0, 0, 1.0, 50.0], **ap),
                  Drift("D", 0.1), Aperture("A", [-4e-3, 4e-3, -3e-3, 3e-3]),
                  Quadrupole("Q", 0.2, 1.0, **ap)]
    ring = Lattice(elems, energy=3.0e9, particle=Particle("electron"), name="apertures")
    n = len(ring)
    every = np.arange(n + 1, dtype=np.uint32)
    beam = _beam(100)
    want = _check(ring, beam, 2, every)
    assert len(set(want["elem"][want["islost"] != 0])) > 3
    rest = ring.particle.rest_energy
    dl = engine.DeviceLattice(ring)
    try:
        for start in range(n):  # turns that start and end inside a record
            for end in (start + 1, min(start + 3, n), n):
                for strict in (True, False):
                    ref, got = beam.copy(order="F"), beam.copy(order="F")
                    po.atpass(ring, ref, 1, start_elem=start, end_elem=end)
                    dl.track(got, 1, None, energy=ring.energy, rest_energy=rest, start_elem=start,
                             end_elem=end, strict=strict)
                    if strict:
                        np.testing.assert_array_equal(got, ref)
                    else:
                        np.testing.assert_allclose(got, ref, rtol=1e-12, atol=1e-12)
    finally:
        dl.close()


@pytest.mark.parametrize("ppt", [1, 2])
@pytest.mark.parametrize("rare", [False, True], ids=["common", "rare"])
def test_wide_particle_leaves_the_others_alone(rare, ppt):
    """A wave whose radiating magnets need the checks takes the rest of the turn in the loop with
    the checks; its other particles get the same bits, with refpt copies and without."""
    q = {"PassMethod": "StrMPoleSymplectic4RadPass"}
    b = {"PassMethod": "BndMPoleSymplectic4RadPass"}
    scale = {"FieldScaling": 1.001} if rare else {}
    elems = [Marker("M")]
    for _ in range(4):
        elems += [Drift("D", 0.3), Quadrupole("Q", 0.4, 1.2, **q, **scale), Drift("D", 0.3),
                  Dipole("B", 1.0, 0.05, 0.0, **b), Sextupole("S", 0.2, 20.0), Drift("D", 0.2),
                  Quadrupole("Q", 0.4, -1.2, **q), Dipole("B", 1.0, 0.05, -0.1, **b, **scale)]
    elems += [RFCavity("RF", 0.0, 1e6, 500e6, 100, 3e9), Drift("D", 0.1)]
    ring = Lattice(elems, energy=3.0e9, particle=Particle("electron"), name="wide")
    rest = ring.particle.rest_energy
    beam = 0.1 * _beam()
    wild = beam.copy(order="F")
    wild[1, 70] = 0.02     # outside at the first magnet
    wild[1, 140], wild[0, 140] = 0.0095, 0.01  # on the way, in another wave
    others = np.ones(beam.shape[1], bool)
    others[[70, 140]] = False
    every = np.arange(len(ring) + 1, dtype=np.uint32)
    dl = engine.DeviceLattice(ring)
    try:
        dl.set_launch_shape(ppt=ppt)
        for refs in (None, every):
            calm, got = beam.copy(order="F"), wild.copy(order="F")
            copies0, _ = dl.track(calm, 3, refs, energy=ring.energy, rest_energy=rest, losses=True)
            copies1, _ = dl.track(got, 3, refs, energy=ring.energy, rest_energy=rest, losses=True)
            np.testing.assert_array_equal(got[:, others], calm[:, others])
            if refs is not None:
                np.testing.assert_array_equal(copies1[:, others], copies0[:, others])
    finally:
        dl.close()
    _check(ring, wild, 3)
    _check(ring, wild, 2, every)
