"""GPU: the program records of the tracking kernel (markers, a plain drift and
an element in one record) against the oracle: every partial turn that starts
or ends inside a record, refpt copies inside records, losses at each part of
one, and inputs that are lost or not finite. Strict build: bit for bit; fast
build: |diff| <= 1e-12 for particles that stay finite, the same loss records."""

import numpy as np
import pytest

from at_amd import engine
from at_amd.lattice import (Aperture, Corrector, Dipole, Drift, Lattice, Marker, Octupole,
                            Particle, Quadrupole, Sextupole, ThinMultipole)
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

RAD_S, RAD_B = "StrMPoleSymplectic4RadPass", "BndMPoleSymplectic4RadPass"


def _ring():
    """Records: [marker, drift, marker...] and every op, one of them misaligned."""
    shifted = Quadrupole("QM", 0.3, 1.1)
    shifted.T1 = np.array([-1e-4, 0.0, 2e-4, 0.0, 0.0, 0.0])
    shifted.T2 = -shifted.T1
    c, s = np.cos(1e-3), np.sin(1e-3)
    roll = np.eye(6)
    roll[0, 0] = roll[1, 1] = roll[2, 2] = roll[3, 3] = c
    roll[0, 2] = roll[1, 3] = s
    roll[2, 0] = roll[3, 1] = -s
    shifted.R1, shifted.R2 = roll, roll.T.copy()
    elems = [Marker("M"), Drift("D", 0.2), Marker("M"), Marker("M"), Quadrupole("Q", 0.4, 1.2),
             Drift("D", 0.3), Aperture("A", [-4e-3, 4e-3, -3e-3, 3e-3]), Drift("D", 0.1),
             Drift("D", 0.2), Corrector("C", 0.0, [1e-5, -2e-5]),
             Corrector("C", 0.1, [1e-5, 2e-5]), Marker("M"), Drift("D", 0.2), shifted,
             Dipole("B", 1.0, 0.05, -0.3, EntranceAngle=0.02, ExitAngle=0.03),
             Sextupole("S", 0.2, 20.0), Octupole("O", 0.1, [0, 0, 0, 0], [0, 0, 0, 300.0]),
             Quadrupole("QR", 0.4, -1.2, PassMethod=RAD_S), Drift("D", 0.3),
             Dipole("BR", 1.0, 0.05, 0.2, PassMethod=RAD_B),
             ThinMultipole("T", [0, 0, 0], [0, 0, 3.0]),
             ThinMultipole("T", [0, 0, 0, 0], [0, 0, 1.0, 50.0]),
             Dipole("BE", 1.0, 0.05, 0.2, EntranceAngle=0.02, ExitAngle=0.03,
                    FringeBendEntrance=2, FringeBendExit=2), Marker("M")]
    return Lattice(elems, energy=6.0e9, particle=Particle("electron"), name="records")


def _beam(n=96):
    r = np.asfortranarray(np.random.default_rng(5).standard_normal((6, n))
                          * np.array([2e-3, 3e-4, 1.5e-3, 2e-4, 1e-3, 1e-3])[:, None])
    r[0, 3] = np.nan        # skipped and lost at the first element
    r[1, 4] = np.inf
    r[0, 5] = 1.5           # |x| > 1
    r[4, 6] = -2.0
    r[:, 7] = [np.nan, 0.1, 0.2, 0.3, 0.4, 0.5]
    r[5, 8] = np.inf
    return r


def _check(ring, dl, beam, nturns, refs, losses, start, end, strict):
    got, ref = beam.copy(order="F"), beam.copy(order="F")
    a = dl.track(got, nturns, refs, energy=ring.energy, rest_energy=ring.particle.rest_energy,
                 losses=losses, start_elem=start, end_elem=end, strict=strict)
    b = po.atpass(ring, ref, nturns, refpts=refs, losses=losses, start_elem=start, end_elem=end)
    what = f"start {start} end {end} losses {losses} strict {strict}"
    (ao, al), (bo, bl) = (a, b) if losses else ((a, None), (b, None))
    if losses:
        for k in ("islost", "turn", "elem"):
            np.testing.assert_array_equal(al[k], bl[k], err_msg=f"{what} {k}")
    if strict:
        np.testing.assert_array_equal(got, ref, err_msg=what)
        np.testing.assert_array_equal(ao, bo, err_msg=what)
        if losses:
            np.testing.assert_array_equal(al["coord"], bl["coord"], err_msg=what)
    else:
        for x, y in ((got, ref), (ao, bo)):
            fine = np.isfinite(y)
            np.testing.assert_array_equal(fine, np.isfinite(x), err_msg=what)
            np.testing.assert_allclose(x[fine], y[fine], rtol=1e-12, atol=1e-12, err_msg=what)


@pytest.mark.parametrize("strict", [True, False], ids=["strict", "fast"])
@pytest.mark.parametrize("losses", [True, False], ids=["losses", "no_losses"])
def test_partial_turns(strict, losses):
    ring = _ring()
    n = len(ring)
    dl = engine.DeviceLattice(ring)
    every = np.arange(n + 1, dtype=np.uint32)
    beam = _beam()
    if not losses:  # at.c leaves an infinite x as it is: elements go on with it
        beam = np.asfortranarray(beam[:, np.isfinite(beam).all(axis=0) | np.isnan(beam[0])])
    try:
        for start in range(n):
            for end in range(start, n + 1):
                for refs in (every, None):
                    if end == 0:
                        continue  # 0 stands for the whole ring
                    _check(ring, dl, beam, 1, refs, losses, start, end, strict)
            _check(ring, dl, beam, 3, None, losses, start, n, strict)
        _check(ring, dl, beam, 3, every, losses, 0, n, strict)
    finally:
        dl.close()
