"""GPU: per-element diffusion matrices against Ohmi's propagation B <- M B M^T + D in
numpy, with whole 6x6 products (the kernel leaves out those with the zeros and ones
of the maps' matrices): straight, curved and exact radiating passes from off-axis
orbits with all coordinates nonzero. Entry i, j is bounded by sqrt(B_ii B_jj); the
kicks of a slice have both signs and leave about a third of their sum, so a few
hundred operations stay below 1e-11 of that."""

import numpy as np
import pytest

from at_amd import engine
from at_amd.lattice import Dipole, Lattice, Multipole, Particle, Quadrupole

pytestmark = pytest.mark.gpu

RE, E0 = 2.8179403205e-15, 510.99895069e-6  # classical electron radius, electron mass in GeV
RAD = 2.0 / 3.0 * RE
DIF = 55.0 / 24.0 / np.sqrt(3.0) * 197.3269804e-18 / E0 * RE
CBRT2 = 2.0 ** (1.0 / 3.0)
DRIFTS = (1.0 / (2.0 * (2.0 - CBRT2)), 0.5 - 1.0 / (2.0 * (2.0 - CBRT2)))
KICKS = (1.0 / (2.0 - CBRT2), 1.0 - 2.0 / (2.0 - CBRT2))
STR, BND, EXACT = ("StrMPoleSymplectic4RadPass", "BndMPoleSymplectic4RadPass",
                   "ExactMultipoleRadPass")


def _field(e, x, y):
    """Field (re, im) and its derivative, coefficient by coefficient."""
    z = complex(x, y)
    c = [complex(b, a) for a, b in zip(e.PolynomA, e.PolynomB)]
    return sum(k * z ** i for i, k in enumerate(c)), sum(i * k * z ** (i - 1)
                                                         for i, k in enumerate(c) if i)


def _drift(r, b, length, exact):
    x, px, y, py, dp, ct = r
    p = 1.0 / (1.0 + dp)
    u, v = px * p, py * p
    m = np.eye(6)
    if exact:
        den = 1.0 - u * u - v * v
        nl = length * p / np.sqrt(den)
        m[0, 1], m[0, 3], m[0, 4] = nl * (1 - v * v) / den, nl * u * v / den, -nl * u / den
        m[2, 1], m[2, 3], m[2, 4] = nl * u * v / den, nl * (1 - u * u) / den, -nl * v / den
        m[5, 1], m[5, 3], m[5, 4] = nl * u / den, nl * v / den, -nl * (u * u + v * v) / den
        path = nl * (1 + dp)
    else:
        nl = length * p
        m[0, 1], m[0, 4], m[2, 3], m[2, 4] = nl, -nl * u, nl, -nl * v
        m[5, 1], m[5, 3], m[5, 4] = nl * u, nl * v, -nl * (u * u + v * v)
        path = 0.5 * nl * p * (px * px + py * py)
    return np.array([x + nl * px, px, y + nl * py, py, dp, ct + path]), m @ b @ m.T


def _kick(r, b, e, length, h, rad, dif):
    x, px, y, py, dp, ct = r
    f, df = _field(e, x, y)
    p = 1.0 / (1.0 + dp)
    u, v = px * p, py * p
    exact = e.PassMethod == EXACT
    if exact:
        b2 = f.imag ** 2 + f.real ** 2 - (f.imag * u + f.real * v) ** 2
        factor = length / p ** 2 / np.sqrt(1 - u * u - v * v)
    else:
        hx, by, bx = 1.0 + h * x, f.real + h, f.imag
        b2 = ((by * hx) ** 2 + (bx * hx) ** 2 + (bx * v - by * u) ** 2) / (hx * hx + u * u + v * v)
        factor = (hx + 0.5 * (u * u + v * v)) / p ** 2 * length
    m = np.eye(6)
    m[1, 0], m[1, 2] = -length * (df.real + h * h), length * df.imag
    m[3, 0], m[3, 2] = length * df.imag, length * df.real
    m[1, 4], m[5, 0] = length * h, length * h
    w = np.array([0.0, u, 0.0, v, 1.0, 0.0])
    d = dif * b2 ** 1.5 * factor / p ** 2 * np.outer(w, w)
    dp1 = dp - rad * b2 * factor
    px1 = u * (1 + dp1) - length * (f.real - (dp - x * h) * h)
    py1 = v * (1 + dp1) + length * f.imag
    return np.array([x, px1, y, py1, dp1, ct + length * h * x]), m @ b @ m.T + d


def _edge(r, b, angle, h):
    m = np.eye(6)
    m[1, 0], m[3, 2] = h * np.tan(angle), -h * np.tan(angle)
    return m @ r, m @ b @ m.T


def _diffusion(e, orbit, energy, rest):
    gamma = energy / rest
    rad, dif = RAD * gamma ** 3, DIF * gamma ** 5
    r, b = np.array(orbit, float), np.zeros((6, 6))
    bend = e.PassMethod == BND
    h = e.BendingAngle / e.Length if bend else 0.0
    step = e.Length / e.NumIntSteps
    if bend:
        r, b = _edge(r, b, e.EntranceAngle, h)
    for _ in range(e.NumIntSteps):
        for d, k in zip((0, 1, 1, 0), (0, 1, 0, None)):
            r, b = _drift(r, b, step * DRIFTS[d], e.PassMethod == EXACT)
            if k is not None:
                r, b = _kick(r, b, e, step * KICKS[k], h, rad, dif)
    if bend:
        r, b = _edge(r, b, e.ExitAngle, h)
    return b


A4, B4 = [1e-3, -0.2, 2.0, 30.0], [2e-3, 0.9, -8.0, 200.0]
ELEMENTS = {
    "quad": Quadrupole("Q", 0.4, 1.2, PassMethod=STR, NumIntSteps=3),
    "multipole": Multipole("M", 0.3, A4, B4, PassMethod=STR, NumIntSteps=4),
    "bend": Dipole("B", 1.0, 0.05, -0.3, PassMethod=BND, EntranceAngle=0.02, ExitAngle=0.03),
    "bend_all": Dipole("B", 1.0, 0.05, 0.0, PassMethod=BND, PolynomA=A4[:3], PolynomB=B4[:3],
                       MaxOrder=2, EntranceAngle=0.02, ExitAngle=0.03, NumIntSteps=5),
    "exact": Multipole("X", 0.3, A4, B4, PassMethod=EXACT, NumIntSteps=2),
}


@pytest.mark.parametrize("kind", ELEMENTS)
def test_dense_products(kind):
    e = ELEMENTS[kind]
    ring = Lattice([e], energy=6.0e9, particle=Particle("electron"), name="one")
    rest = ring.particle.rest_energy
    dl = engine.DeviceLattice(ring)
    rng = np.random.default_rng(11)
    try:
        for _ in range(6):
            orbit = rng.normal(0.0, [1e-3, 3e-3, 5e-4, 2e-3, 2e-2, 1e-3])
            got = dl.diffusion_matrices(orbit.reshape(6, 1), ring.energy, rest)[0]
            want = _diffusion(e, orbit, ring.energy, rest)
            assert np.count_nonzero(want) >= 30  # all but the row and column of an unmoved ct
            scale = np.sqrt(np.abs(np.outer(np.diag(want), np.diag(want))))
            assert (np.abs(got - want) <= 1e-11 * scale).all()
    finally:
        dl.close()
