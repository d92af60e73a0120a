"""GPU: refpt copies of whole and of partly filled waves (a lane per particle, 64 to
a wave, and two particles per lane): beams around a wave's size, particles that are
lost on the way in some waves only, an input that is not finite. Strict build: bit for
bit the oracle's copies; fast build: bit for bit those of each particle alone."""

import numpy as np
import pytest

from at_amd import engine
from at_amd.lattice import Aperture, Drift, Lattice, Marker, Particle, Quadrupole
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def _ring():
    elems = []
    for _ in range(12):  # more than one word of 32 elements
        elems += [Drift("D", 0.5), Quadrupole("Q", 0.3, 1.5), Marker("M"), Drift("D", 0.5),
                  Quadrupole("Q", 0.3, -1.5)]
    elems.insert(31, Aperture("A", [-3e-3, 3e-3, -3e-3, 3e-3]))
    return Lattice(elems, energy=3.0e9, particle=Particle("electron"), name="waves")


@pytest.mark.parametrize("ppt", [1, 2])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 127, 128, 129, 257])
def test_copies_of_waves(n, ppt):
    ring = _ring()
    ne = len(ring)
    every = np.arange(ne + 1, dtype=np.uint32)
    beam = np.asfortranarray(np.random.default_rng(4).standard_normal((6, n))
                             * np.array([5e-4, 1e-4, 5e-4, 1e-4, 1e-3, 1e-3])[:, None])
    if n > 100:  # the first wave loses particles, the others lose none
        beam[0, 7], beam[0, 11], beam[2, 30] = 2.9e-2, np.nan, 2.0
    dl = engine.DeviceLattice(ring)
    dl.set_launch_shape(ppt=ppt)
    kw = {"energy": ring.energy, "rest_energy": ring.particle.rest_energy, "losses": True}
    try:
        ref = beam.copy(order="F")
        want, lost = po.atpass(ring, ref, 3, refpts=every, losses=True)
        got = beam.copy(order="F")
        have, hlost = dl.track(got, 3, every, strict=True, **kw)
        np.testing.assert_array_equal(got, ref)
        np.testing.assert_array_equal(have, want)
        for k in ("islost", "turn", "elem", "coord"):
            np.testing.assert_array_equal(hlost[k], lost[k], err_msg=k)
        fast = beam.copy(order="F")
        have, _ = dl.track(fast, 3, every, **kw)
        for p in sorted({0, 7, 11, 30, 62, 63, 64, 126, 127, 128, n - 1} & set(range(n))):
            one = np.asfortranarray(beam[:, p:p + 1])
            alone, _ = dl.track(one, 3, every, **kw)
            np.testing.assert_array_equal(fast[:, p], one[:, 0])
            np.testing.assert_array_equal(have[:, p], alone[:, 0])
    finally:
        dl.close()
