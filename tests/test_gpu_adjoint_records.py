"""GPU: the adjoint of a magnet by its record (misaligned by shifts and rolls or not,
by the form of its field) against the adjoint by its header, which zero coefficients
up to MaxOrder 4 select, and against central differences of the oracle. The two
adjoints differ in rounding only: a few hundred operations on entries up to the
matrix's largest, 1e-12 of it."""

import numpy as np
import pytest

from at_amd import engine
from at_amd import lattice as L
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

ENERGY = 6.0e9
POINTS = np.array([[1e-3, 2e-4, -5e-4, 1e-4, 1e-3, 1e-3], [-2e-3, 1e-5, 8e-4, -3e-4, -5e-3, 0.0]])
KINDS = {
    "quad": (L.Quadrupole, ("Q", 0.5, 1.3), {"NumIntSteps": 10}, 1),
    "quad1": (L.Quadrupole, ("Q", 0.5, 1.3), {"NumIntSteps": 1}, 1),
    "sext": (L.Sextupole, ("S", 0.2, 35.0), {"NumIntSteps": 3}, 2),
    "steerer": (L.Sextupole, ("S", 0.2, 35.0), {"NumIntSteps": 10, "PolynomB": [1e-3, 0.0, 35.0],
                                                "PolynomA": [-2e-3, 0.0, 0.0]}, 2),
    "steerer_b0": (L.Sextupole, ("S", 0.2, 35.0), {"NumIntSteps": 2, "PolynomB": [1e-3, 0.0, 35.0],
                                                   "PolynomA": [-2e-3, 0.0, 0.0]}, 0),
    "oct": (L.Octupole, ("O", 0.1, [0, 0, 0, 0], [0, 0, 0, 500.0]), {"NumIntSteps": 4}, 3),
    "bend": (L.Dipole, ("B", 1.0, 0.03, 0.0), {"EntranceAngle": 0.015, "ExitAngle": 0.01}, 1),
    "bend_grad": (L.Dipole, ("B", 1.0, 0.03, -0.9), {"EntranceAngle": 0.015, "ExitAngle": 0.01,
                                                     "NumIntSteps": 10}, 1),
    "all": (L.Quadrupole, ("Q", 0.4, 1.2), {"PolynomA": [1e-3, -0.2], "PolynomB": [2e-3, 0.9]}, 1),
}


def _rot(psi):
    c, s = np.cos(psi), np.sin(psi)
    r = np.eye(6)
    r[0, 0] = r[1, 1] = r[2, 2] = r[3, 3] = c
    r[0, 2] = r[1, 3] = s
    r[2, 0] = r[3, 1] = -s
    return r


def _magnet(kind, how):
    make, args, kw, coeff = KINDS[kind]
    m = make(*args, **kw)
    if how in ("shift", "all"):
        m.T1, m.T2 = np.array([1e-4, 1e-5, -2e-4, 0, 0, 0]), np.array([-1e-4, 0, 2e-4, 2e-5, 0, 0])
    if how in ("r1", "all"):
        m.R1 = _rot(0.02)
    if how in ("r2", "all"):
        m.R2 = _rot(-0.03)
    return m, coeff


def _adjoint(elems, which, coeff):
    """Rows of the Jacobian of the elements at each point, and the gradients."""
    import torch

    lat = L.Lattice(elems, energy=ENERGY, particle="electron")
    rest = lat.particle.rest_energy
    dl = engine.DeviceLattice(lat)
    n = 6 * len(POINTS)
    dev = torch.device("cuda:0")
    states = torch.empty((2, n, 6), dtype=torch.float64, device=dev)
    states[:] = torch.tensor(np.repeat(POINTS, 6, axis=0), device=dev)
    stream = torch.cuda.current_stream().cuda_stream
    slots = np.full(len(elems), -1, np.int32)
    slots[which] = 0
    coeffs = np.full(len(elems), 0, np.int32)
    coeffs[which] = coeff
    grads = []
    try:
        dl.track_device(states[1].data_ptr(), n, 1, energy=ENERGY, rest_energy=rest, stream=stream)
        for i in range(6):  # the gradient of each coordinate, summed over the points
            lam = torch.zeros((n, 6), dtype=torch.float64, device=dev)
            lam[:, i] = 1.0
            g = torch.zeros(1, dtype=torch.float64, device=dev)
            dl.adjoint(states.data_ptr(), 1, 0, n, ENERGY, rest, lam.data_ptr(), slots, coeffs,
                       g.data_ptr(), 1, stream=stream)
            torch.cuda.synchronize()
            grads.append((lam.cpu().numpy()[::6], float(g) / 6))
    finally:
        dl.close()
    return np.array([g[0] for g in grads]).transpose(1, 0, 2), np.array([g[1] for g in grads])


def _oracle(elems, r6):
    lat = L.Lattice(elems, energy=ENERGY, particle="electron")
    a = np.asfortranarray(r6.reshape(6, 1).copy())
    po.atpass(lat, a, 1)
    return a[:, 0]


@pytest.mark.parametrize("how", ["none", "shift", "r1", "r2", "all"])
@pytest.mark.parametrize("kind", KINDS)
def test_record_equals_header(kind, how):
    m, coeff = _magnet(kind, how)
    elems = [L.Drift("D", 0.3), m, L.Drift("D", 0.2)]
    rows, grad = _adjoint(elems, 1, coeff)
    by_header, _ = _magnet(kind, how)
    for name in ("PolynomA", "PolynomB"):
        poly = np.zeros(5)
        poly[:len(getattr(m, name))] = getattr(m, name)
        setattr(by_header, name, poly)
    by_header.MaxOrder = 4
    rows_h, grad_h = _adjoint([L.Drift("D", 0.3), by_header, L.Drift("D", 0.2)], 1, coeff)
    np.testing.assert_allclose(rows, rows_h, rtol=0, atol=1e-12 * max(1.0, np.abs(rows_h).max()))
    np.testing.assert_allclose(grad, grad_h, rtol=0, atol=1e-12 * np.abs(grad_h).max())
    for ip, r6 in enumerate(POINTS):
        h = 1e-7
        fd = np.array([(_oracle(elems, r6 + h * d) - _oracle(elems, r6 - h * d)) / (2 * h)
                       for d in np.eye(6)]).T
        # central differences: rounding 1e-16 / 1e-7, curvature below 1e4 x 1e-14
        np.testing.assert_allclose(rows[ip], fd, rtol=0, atol=2e-8 * max(1.0, np.abs(fd).max()))
