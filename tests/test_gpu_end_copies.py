"""GPU: refpt copies at the end of the ring only, which the kernel without copies
inside a turn makes, against the oracle: several turns with losses on the way,
partial turns, particles that are lost or not finite at the start, both layouts of
lanes. Strict build: bit for bit; fast build: as the same call with copies at every
element, bit for bit."""

import numpy as np
import pytest

from at_amd import engine
from at_amd.lattice import Aperture, Dipole, Drift, Lattice, Marker, Particle, Quadrupole
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def _ring():
    elems = [Marker("M")]
    for _ in range(11):
        elems += [Drift("D", 0.5), Quadrupole("Q", 0.3, 1.5), Drift("D", 0.5),
                  Quadrupole("Q", 0.3, -1.5)]
    elems += [Aperture("A", [-4e-3, 4e-3, -3e-3, 3e-3]),
              Dipole("B", 0.5, 0.02, 0.0, PassMethod="BndMPoleSymplectic4RadPass")]
    return Lattice(elems, energy=3.0e9, particle=Particle("electron"), name="ends")


def _beam(n):
    r = np.asfortranarray(np.random.default_rng(9).standard_normal((6, n))
                          * np.array([1.5e-3, 2e-4, 1.2e-3, 2e-4, 1e-3, 1e-3])[:, None])
    r[0, 3 % n], r[1, 5 % n], r[0, 7 % n] = np.nan, np.inf, 1.5
    r[1, 9 % n] = 0.02
    return r


@pytest.mark.parametrize("losses", [True, False], ids=["losses", "no_losses"])
@pytest.mark.parametrize("ppt", [1, 2])
@pytest.mark.parametrize("n", [1, 64, 200, 1000])
def test_end_copies(n, ppt, losses):
    ring = _ring()
    ne = len(ring)
    rest = ring.particle.rest_energy
    last = np.array([ne], np.uint32)
    every = np.arange(ne + 1, dtype=np.uint32)
    dl = engine.DeviceLattice(ring)
    dl.set_launch_shape(ppt=ppt)
    kw = {"energy": ring.energy, "rest_energy": rest, "losses": losses}
    try:
        for turns, start, end in ((1, 0, ne), (6, 0, ne), (3, 7, ne), (1, 2, 9)):
            beam = _beam(n)
            if not losses:
                beam = np.asfortranarray(beam[:, np.isfinite(beam).all(axis=0)])
                if beam.shape[1] == 0:
                    continue
            ref = beam.copy(order="F")
            want = po.atpass(ring, ref, turns, refpts=last, losses=losses, start_elem=start,
                             end_elem=end)
            got = beam.copy(order="F")
            have = dl.track(got, turns, last, start_elem=start, end_elem=end, strict=True, **kw)
            wc, hc = (want[0], have[0]) if losses else (want, have)
            assert hc.shape == wc.shape and hc.shape[2:] == (1, turns)
            np.testing.assert_array_equal(got, ref)
            np.testing.assert_array_equal(hc, wc)
            if losses:
                for k in ("islost", "turn", "elem", "coord"):
                    np.testing.assert_array_equal(have[1][k], want[1][k], err_msg=k)
            fast, both = beam.copy(order="F"), beam.copy(order="F")
            a = dl.track(fast, turns, last, start_elem=start, end_elem=end, **kw)
            b = dl.track(both, turns, every, start_elem=start, end_elem=end, **kw)
            ac, bc = (a[0], b[0]) if losses else (a, b)
            np.testing.assert_array_equal(fast, both)
            if start == 0 and end == ne:
                np.testing.assert_array_equal(ac[:, :, 0], bc[:, :, -1])
    finally:
        dl.close()
