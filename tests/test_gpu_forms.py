"""GPU: the kicks of thick multipoles by the form of their field (one leading
coefficient, that and a dipole, none, all) against the oracle, at slice counts
around the unrolled loop's, misaligned or not, with particles outside the ranges
of the fast build's series (angles above 10 mrad, radiated fractions above 2e-6
per kick) and particles that overflow inside an element. Strict build: bit for
bit; fast build: a magnet's few hundred roundings of coordinates below 1 stay
below 1e-12, and the loss records are the same."""

import numpy as np
import pytest

from at_amd import engine
from at_amd.lattice import Dipole, Drift, Lattice, Octupole, Particle, Quadrupole, Sextupole
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

RAD_S, RAD_B = "StrMPoleSymplectic4RadPass", "BndMPoleSymplectic4RadPass"
A2, B2 = [0.01, -0.2], [0.002, 0.9]


def _magnet(kind, rad):
    s = {"PassMethod": RAD_S} if rad else {}
    b = {"PassMethod": RAD_B} if rad else {}
    edges = {"EntranceAngle": 0.02, "ExitAngle": 0.03}
    if kind == "quad":
        return Quadrupole("Q", 0.4, -1.2, **s)
    if kind == "quad_all":
        return Quadrupole("Q", 0.4, 1.2, PolynomA=A2, PolynomB=B2, **s)
    if kind == "bend":
        return Dipole("B", 1.0, 0.1, 0.0, **edges, **b)
    if kind == "bend_grad":
        return Dipole("B", 1.0, 0.1, -0.3, **edges, **b)
    if kind == "bend_all":
        return Dipole("B", 1.0, 0.1, 0.0, PolynomA=A2, PolynomB=B2, **edges, **b)
    if kind == "sext":
        return Sextupole("S", 0.2, 20.0, **s)
    if kind == "sext_steerer":
        return Sextupole("S", 0.2, 20.0, PolynomB=[1e-4, 0.0, 20.0], PolynomA=[-2e-4, 0.0, 0.0], **s)
    if kind == "sext_all":
        return Sextupole("S", 0.2, 20.0, PolynomB=[1e-4, 0.1, 20.0], PolynomA=[0.0, 0.1, 3.0], **s)
    if kind == "oct":
        return Octupole("O", 0.1, [0, 0, 0, 0], [0, 0, 0, 300.0], **s)
    return Octupole("O", 0.1, [1e-5, 0, 0, 7.0], [0, 0.1, 0, 300.0], **s)


KINDS = ["quad", "quad_all", "bend", "bend_grad", "bend_all", "sext", "sext_steerer", "sext_all",
         "oct", "oct_all"]


@pytest.mark.parametrize("rad", [False, True], ids=["plain", "rad"])
@pytest.mark.parametrize("kind", KINDS)
def test_form(kind, rad):
    c, s = np.cos(1e-3), np.sin(1e-3)
    roll = np.eye(6)
    roll[0, 0] = roll[1, 1] = roll[2, 2] = roll[3, 3] = c
    roll[0, 2] = roll[1, 3] = s
    roll[2, 0] = roll[3, 1] = -s
    elems = []
    for n in (1, 2, 3, 10):
        m = _magnet(kind, rad)
        m.NumIntSteps = n
        elems += [Drift("D", 0.1), m]
    moved = _magnet(kind, rad)
    moved.T1, moved.T2 = np.array([1e-4, 0, -2e-4, 0, 0, 0]), np.array([-1e-4, 0, 2e-4, 0, 0, 0])
    moved.R1, moved.R2 = roll, roll.T.copy()
    # 40 GeV: a bend's kick radiates more than 2e-6 of the energy
    for energy in (3.0e9, 4.0e10):
        ring = Lattice(elems + [Drift("D", 0.1), moved], energy=energy, particle=Particle("electron"),
                       name="forms")
        n = 200
        beam = np.asfortranarray(np.random.default_rng(3).standard_normal((6, n))
                                 * np.array([1e-3, 2e-4, 1e-3, 2e-4, 1e-3, 1e-3])[:, None])
        beam[1, 70:74] = [0.02, -0.03, 0.05, 0.011]  # wide angles, in one wave
        beam[3, 72:76] = [0.02, 0.03, -0.05, 0.011]
        beam[0, 150] = 0.99  # beyond any aperture: overflows in the strong multipoles
        beam[2, 151] = -0.95
        rest = ring.particle.rest_energy
        dl = engine.DeviceLattice(ring)
        try:
            ref = beam.copy(order="F")
            _, want = po.atpass(ring, ref, 2, losses=True)
            for strict in (True, False):
                got = beam.copy(order="F")
                _, have = dl.track(got, 2, None, energy=ring.energy, rest_energy=rest, losses=True,
                                   strict=strict)
                for k in ("islost", "turn", "elem"):
                    np.testing.assert_array_equal(have[k], want[k], err_msg=f"{strict} {k}")
                if strict:
                    np.testing.assert_array_equal(got, ref)
                else:
                    np.testing.assert_array_equal(np.isfinite(got), np.isfinite(ref))
                    fine = np.isfinite(ref)
                    np.testing.assert_allclose(got[fine], ref[fine], rtol=1e-12, atol=1e-12)
        finally:
            dl.close()
