"""GPU: the tracking loss without a backward to come (torch.no_grad, or strengths
that need no gradient): one launch per checkpoint block, as nothing is kept for
backward, and the same loss bit for bit."""

import numpy as np
import pytest

from at_amd import engine
from at_amd.adjoint import Problem, TrackingLoss
from at_amd.lattice import Quadrupole
from at_amd.workloads import fodo_ring, gaussian_beam

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nturns,blocks", [(1, 1), (8, 1), (11, 2), (24, 3)])
def test_launches(monkeypatch, nturns, blocks):
    import torch

    ring = fodo_ring()
    problem = Problem(ring, [(i, 1) for i, e in enumerate(ring) if isinstance(e, Quadrupole)])
    theta = torch.tensor(problem.initial_strengths(), dtype=torch.float64, requires_grad=True)
    beam = torch.from_numpy(np.ascontiguousarray(gaussian_beam(100, seed=3).T)).cuda()
    calls = []
    launch = engine.track_batch

    def counted(*args, **kwargs):
        calls.append(1)
        return launch(*args, **kwargs)

    monkeypatch.setattr(engine, "track_batch", counted)
    with torch.no_grad():
        quiet = TrackingLoss.apply(problem, theta, beam, nturns)
    assert len(calls) == blocks
    calls.clear()
    detached = TrackingLoss.apply(problem, theta.detach(), beam, nturns)
    assert len(calls) == blocks
    loss = TrackingLoss.apply(problem, theta, beam, nturns)
    loss.backward()
    assert theta.grad is not None and float(theta.grad.abs().max()) > 0
    assert float(quiet) == float(detached) == float(loss.detach())
