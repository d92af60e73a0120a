"""Performance cases of the tracking framework, through its public entry points.

Each case is one call, or one short sequence of calls, that a user's program
makes: reading an orbit with one particle, tracking beams from host arrays
and from device buffers, dynamic-aperture grids of many error realisations in
one launch, a served batch of requests, a gradient of a tracking loss, linear
optics and the matrices of a radiation envelope. Lattices are the
framework's own workloads: ``fodo_ring`` (320 elements, no radiation) and
``large_ring`` (2,241 elements, radiating bends and quadrupoles, one cavity,
apertures), with seeded corrector kicks or seeded magnet errors.

``exact`` recomputes the outputs with the element maps written out in numpy
(FP64), without the engine, where that takes seconds.
"""

import math

import numpy as np
import torch

from at_amd import engine, flops, physics
from at_amd.adjoint import Problem, TrackingLoss
from at_amd.batch import track_batch
from at_amd.lattice import Quadrupole, Sextupole
from at_amd.serving import Request, Server
from at_amd.tracking import lattice_track
from at_amd.workloads import (corrected_realisations, da_polar_grid, fodo_ring, gaussian_beam,
                              large_ring)

C_LIGHT = 2.99792458e8
MATRIX_STEP = 3.0e-8


def listed():
    return [
        # one particle once around a small ring, the coordinates kept at every
        # element: reading an orbit; bound by the call and by one lane's chain
        {"name": "orbit_1", "kind": "host", "ring": "fodo", "n": 1, "turns": 1, "refpts": True},
        # an ordinary beam in a small ring from host arrays with a loss map,
        # the plain-tracking workload
        {"name": "fodo_4096", "kind": "host", "ring": "fodo", "n": 4096, "turns": 8,
         "refpts": False},
        # the first tracking call on a lattice: the call builds the device
        # lattice from the element objects
        {"name": "first_call_1000", "kind": "first", "n": 1000, "turns": 1},
        # a beam that leaves most of the device idle: one GPU's share of a
        # beam, or a served request, with a ragged size
        {"name": "beam_24001", "kind": "device", "n": 24001, "turns": 8, "strict": False,
         "soa": True},
        # the headline workload's beam for a few turns
        {"name": "beam_262144", "kind": "device", "n": 262144, "turns": 8, "strict": False,
         "soa": False},
        # the build that keeps the reference operation order
        {"name": "strict_32003", "kind": "device", "n": 32003, "turns": 2, "strict": True,
         "soa": False},
        # turn-by-turn data: the beam copied at every element, the
        # bandwidth-heavy option
        {"name": "monitors_8191", "kind": "monitors", "n": 8191, "turns": 1},
        # dynamic aperture of corrected error realisations, one launch with
        # the survivors repacked: on every second ring the whole grid, a third
        # of which is lost in its 4 turns, on the others the stable core for
        # longer (points at the edge of stability amplify a rounding
        # difference a thousandfold per turn, so they run few turns)
        {"name": "aperture_16", "kind": "aperture", "rings": 16, "nmin": 1000, "nmax": 16000,
         "turns": 16},
        # a queue of requests of uneven sizes through the server
        {"name": "serve_8", "kind": "serve", "rings": 4, "requests": 8, "nmin": 2000,
         "nmax": 40000},
        # forward and backward: gradient of a tracking loss with respect to
        # every quadrupole and sextupole strength
        {"name": "gradient_4096", "kind": "gradient", "n": 4096, "turns": 8},
        # closed orbit at every element and the transfer matrices there
        {"name": "optics", "kind": "optics", "cells": 32},
        # transfer and diffusion matrix of every element, as an envelope
        # calculation reads them
        {"name": "envelope", "kind": "envelope", "cells": 32},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["host", "host", "first", "device", "device", "device", "monitors",
                       "aperture", "serve", "gradient", "optics", "envelope"])
    if kind == "host":
        return {"kind": kind, "ring": rng.choice(["fodo", "large"]), "n": _log_int(rng, 1, 8000),
                "turns": rng.randint(1, 8), "refpts": False}
    if kind == "first":
        return {"kind": kind, "n": _log_int(rng, 1, 4000), "turns": rng.randint(1, 2)}
    if kind == "device":
        strict = rng.random() < 0.25
        return {"kind": kind, "n": _log_int(rng, 64, 80000 if strict else 262144),
                "turns": rng.randint(1, 8), "strict": strict, "soa": rng.random() < 0.3}
    if kind == "monitors":
        return {"kind": kind, "n": _log_int(rng, 64, 8191), "turns": 1}
    if kind == "aperture":
        return {"kind": kind, "rings": rng.randint(2, 16), "nmin": 1000,
                "nmax": _log_int(rng, 2000, 16000), "turns": rng.randint(2, 16)}
    if kind == "serve":
        return {"kind": kind, "rings": 4, "requests": rng.randint(2, 8), "nmin": 2000,
                "nmax": _log_int(rng, 5000, 40000)}
    if kind == "gradient":
        return {"kind": kind, "n": _log_int(rng, 64, 4096), "turns": rng.randint(1, 8)}
    return {"kind": kind, "cells": rng.randint(3, 32)}


# --- the lattices and inputs of a case --------------------------------------

def _ring(case, seed):
    kind = case["kind"]
    if kind == "host" and case["ring"] == "fodo":
        return fodo_ring()
    if kind in ("gradient", "optics"):
        return large_ring({"corrector_seed": seed}, radiation=False, cavity=kind == "gradient",
                          ncells=case.get("cells"))
    return large_ring({"corrector_seed": seed}, ncells=case.get("cells"))


def _beam(case, seed):
    ring = case.get("ring", "large")
    return gaussian_beam(case["n"], seed=seed, scale=1.0 if ring == "fodo" else 5.0)


def _grids(case, seed):
    """Grids of uneven sizes (the same for every seed), the launch angles spread by the seed."""
    rng = np.random.default_rng(seed)
    out = []
    sizes = np.random.default_rng(7).integers(case["nmin"], case["nmax"] + 1, case["rings"])
    for i, n in enumerate(sizes):
        whole = i % 2 == 0
        g = da_polar_grid(int(n), 15e-3 if whole else 5e-3, 6e-3 if whole else 2e-3, (0.0,))
        g[1] += 1e-6 * rng.standard_normal(g.shape[1])
        out.append(g)
    return out


def _requests(case, seed):
    """Requests of log-uniform sizes (the same for every seed), grids and beams in turn."""
    sizes = np.random.default_rng(7)
    rng = np.random.default_rng(seed)
    out = []
    for i in range(case["requests"]):
        n = int(round(math.exp(sizes.uniform(math.log(case["nmin"]), math.log(case["nmax"])))))
        if i % 2:
            parts, kind = gaussian_beam(n, seed=seed + i, scale=5.0), "track"
        else:
            parts, kind = da_polar_grid(n, deltas=(0.0,)), "da"
        parts[1] += 1e-6 * rng.standard_normal(n)
        out.append(Request(i, i % case["rings"], parts, (4, 16)[i % 2], kind=kind))
    return out


def _orbits(nelem, seed):
    """Orbits at the entrance of every element, as an orbit search returns them."""
    sigma = np.array([1e-4, 1e-5, 1e-4, 1e-5, 1e-4, 1e-4])
    return np.asfortranarray(sigma[:, None]
                             * np.random.default_rng(seed).standard_normal((6, nelem)))


def _on_gpu(beam, soa):
    """(6, N) host beam as the device buffer that a program keeps: (N, 6), or (6, N) planes."""
    return torch.from_numpy(np.ascontiguousarray(beam if soa else beam.T)).cuda()


def _loss_buffers(n):
    return (torch.empty(n, dtype=torch.uint8, device="cuda"),
            torch.empty(n, dtype=torch.int32, device="cuda"),
            torch.empty(n, dtype=torch.int32, device="cuda"),
            torch.empty((n, 6), dtype=torch.float64, device="cuda"))


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case, "kind": kind}
    if kind in ("aperture", "serve"):
        st["rings"] = corrected_realisations(large_ring(), case["rings"])
        st["energy"] = st["rings"][0].energy
        st["rest"] = st["rings"][0].particle.rest_energy
        handles = [engine.DeviceLattice(r) for r in st["rings"]]
        if kind == "serve":
            st["server"] = Server(handles, energy=st["energy"], rest_energy=st["rest"])
            st["requests"] = _requests(case, seed)
        else:
            st["handles"] = handles
            st["turns"] = [(case["turns"] if i % 2 else min(4, case["turns"]), 0)
                           for i in range(case["rings"])]
            st["beams"] = [_on_gpu(g, False) for g in _grids(case, seed)]
        return st
    ring = st["ring"] = _ring(case, seed)
    st["energy"], st["rest"] = ring.energy, ring.particle.rest_energy
    if kind == "host":
        st["lat"] = engine.DeviceLattice(ring)
        st["beam"] = _beam(case, seed)
        st["refs"] = np.arange(len(ring) + 1, dtype=np.uint32) if case["refpts"] else None
    elif kind == "first":
        st["beam"] = _beam(case, seed)
    elif kind in ("device", "monitors"):
        n = case["n"]
        st["lat"] = engine.DeviceLattice(ring)
        st["beam"] = _on_gpu(_beam(case, seed), case.get("soa", False))
        if kind == "monitors":
            st["refs"] = np.arange(len(ring) + 1, dtype=np.uint32)
            st["copies"] = torch.empty((case["turns"], len(ring) + 1, n, 6), dtype=torch.float64,
                                       device="cuda")
        else:
            st["lost"] = _loss_buffers(n)
    elif kind == "gradient":
        params = [(i, 2 if isinstance(e, Sextupole) else 1) for i, e in enumerate(ring)
                  if isinstance(e, (Quadrupole, Sextupole))]
        st["problem"] = Problem(ring, params)
        st["theta"] = torch.tensor(st["problem"].initial_strengths(), dtype=torch.float64,
                                   requires_grad=True)
        st["beam"] = _on_gpu(gaussian_beam(case["n"], seed=seed), False)
    elif kind == "envelope":
        st["lat"] = engine.DeviceLattice(ring)
        st["orbits"] = _orbits(len(ring), seed)
    return st


def run(st):
    kind, case = st["kind"], st["case"]
    stream = torch.cuda.current_stream().cuda_stream
    if kind == "host":
        r = st["beam"].copy(order="F")
        copies, loss = st["lat"].track(r, case["turns"], st["refs"], energy=st["energy"],
                                       rest_energy=st["rest"], losses=True)
        return {"r": r, "copies": copies, "loss": loss}
    if kind == "first":
        out, param, data = lattice_track(st["ring"], st["beam"], case["turns"], losses=True)
        m = data["loss_map"]
        return {"out": out, "r": param["rout"], "islost": m.islost, "turn": m.turn,
                "elem": m.elem, "coord": m.coord}
    if kind == "device":
        r = st["beam"].clone()
        st["lat"].track_device(r.data_ptr(), case["n"], case["turns"], energy=st["energy"],
                               rest_energy=st["rest"], losses=True,
                               loss_ptrs=tuple(b.data_ptr() for b in st["lost"]), stream=stream,
                               strict=case["strict"], soa=case["soa"])
        flag, turn, elem, coord = st["lost"]
        return {"r": r, "flag": flag, "turn": turn, "elem": elem, "coord": coord}
    if kind == "monitors":
        r = st["beam"].clone()
        st["lat"].track_device(r.data_ptr(), case["n"], case["turns"], refpts=st["refs"],
                               rout_ptr=st["copies"].data_ptr(), energy=st["energy"],
                               rest_energy=st["rest"], stream=stream)
        return {"r": r, "copies": st["copies"]}
    if kind == "aperture":
        beams = [b.clone() for b in st["beams"]]
        maps = track_batch(st["handles"], beams, 0, item_turns=st["turns"], energy=st["energy"],
                           rest_energy=st["rest"], stream=stream, repack=True)
        torch.cuda.current_stream().synchronize()
        maps = [m.to_host() for m in maps]
        return {"r": torch.cat(beams), "coord": np.concatenate([m["coord"] for m in maps], 1),
                **{k: np.concatenate([m[k] for m in maps]) for k in ("islost", "turn", "elem")}}
    if kind == "serve":
        results, _ = st["server"].run(st["requests"], realtime=False)
        return [{"r": q.particles, **q.lost} for q in results]
    if kind == "gradient":
        loss = TrackingLoss.apply(st["problem"], st["theta"], st["beam"], case["turns"])
        (grad,) = torch.autograd.grad(loss, st["theta"])
        return {"loss": loss.detach(), "grad": grad}
    if kind == "optics":
        orbit, orbits = physics.find_orbit4(st["ring"], 0.0, range(len(st["ring"]) + 1))
        m44, mats = physics.find_m44(st["ring"], 0.0, range(len(st["ring"]) + 1), orbit=orbit,
                                     keep_lattice=True)
        return {"orbit": orbit, "orbits": orbits, "m44": m44, "mats": mats}
    mats = st["lat"].element_matrices(st["orbits"], MATRIX_STEP, st["energy"], st["rest"])
    diff = st["lat"].diffusion_matrices(st["orbits"], st["energy"], st["rest"])
    return {"mats": mats, "diff": diff}


def work(case):
    """Bytes and FP64 operations of one pass by the map sequence (flops.py). Of
    a whole dynamic-aperture grid two thirds of the particles are counted."""
    kind = case["kind"]
    if kind in ("aperture", "serve"):
        ring = large_ring()
        ops = float(flops.lattice_flops(ring).sum()) + 300.0 * 704
        if kind == "aperture":
            n = 0.5 * (case["nmin"] + case["nmax"]) * case["rings"]
            turns = 0.5 * (case["turns"] + 0.67 * min(4, case["turns"]))
            return {"bytes": 153.0 * n, "flops": ops * n * turns}
        n = case["requests"] * (case["nmax"] - case["nmin"]) / math.log(case["nmax"] / case["nmin"])
        return {"bytes": 201.0 * n, "flops": ops * n * 0.5 * (16 + 0.67 * 4)}
    ring = _ring(case, 1)
    ops = float(flops.lattice_flops(ring).sum())
    if kind == "optics":
        # about four searches and one probe of 9 copies; the probe's copies are kept
        return {"bytes": 48.0 * 10 * len(ring), "flops": 46 * ops}
    if kind == "envelope":
        return {"bytes": 8.0 * (6 + 72) * len(ring), "flops": 12 * ops + 10.0 * ops}
    n, t = case["n"], case["turns"]
    data = 96.0 * n + (57.0 * n if kind != "gradient" else 0)
    if kind == "monitors" or case.get("refpts"):
        data += 48.0 * n * t * (len(ring) + 1)
    return {"bytes": data, "flops": ops * n * t * (3.0 if kind == "gradient" else 1.0)}


# --- the same outputs in numpy ------------------------------------------------

def _slices():
    c = 2.0 ** (1.0 / 3.0)
    d1 = 1.0 / (2.0 * (2.0 - c))
    k1 = 1.0 / (2.0 - c)
    return (d1, 0.5 - d1, 0.5 - d1, d1), (k1, 1.0 - 2.0 * k1, k1)


def _drift(r, length):
    p = 1.0 + r[4]
    r[0] += length * r[1] / p
    r[2] += length * r[3] / p
    r[5] += 0.5 * length * (r[1] * r[1] + r[3] * r[3]) / (p * p)


def _field(r, e):
    z = r[0] + 1j * r[2]
    n = e.MaxOrder
    f = np.full(z.shape, e.PolynomB[n] + 1j * e.PolynomA[n])
    for k in range(n - 1, -1, -1):
        f = f * z + (e.PolynomB[k] + 1j * e.PolynomA[k])
    return f.real, f.imag


def _kick(r, e, length, h, rad):
    re, im = _field(r, e)
    x, dp = r[0].copy(), r[4].copy()
    if rad:
        p = 1.0 + dp
        xp, yp = r[1] / p, r[3] / p
        hx = 1.0 + x * h
        by = re + h
        cross = im * yp - by * xp
        b2 = ((by * hx) ** 2 + (im * hx) ** 2 + cross * cross) / (hx * hx + xp * xp + yp * yp)
        r[4] -= rad * b2 * (hx + 0.5 * (xp * xp + yp * yp)) * p * p * length
        r[1] = xp * (1.0 + r[4])
        r[3] = yp * (1.0 + r[4])
    r[1] -= length * (re - (dp - x * h) * h)
    r[3] += length * im
    r[5] += length * h * x


def _element(r, e, gamma, period, turn):
    """One element for an array of particles (6, n), none of them lost."""
    name = e.PassMethod
    if getattr(e, "R1", None) is not None:
        raise NotImplementedError("misaligned elements")
    if name == "DriftPass":
        _drift(r, e.Length)
    elif name == "AperturePass":
        a = e.Limits
        out = (r[0] < a[0]) | (r[0] > a[1]) | (r[2] < a[2]) | (r[2] > a[3])
        r[5, out] = np.inf
    elif name == "CorrectorPass":
        kx, ky = e.KickAngle
        if e.Length:
            p = 1.0 + r[4]
            q = (kx * kx + ky * ky) / 3.0 + r[1] * (r[1] + kx) + r[3] * (r[3] + ky)
            r[5] += 0.5 * e.Length * q / (p * p)
            r[0] += e.Length * (r[1] + 0.5 * kx) / p
            r[2] += e.Length * (r[3] + 0.5 * ky) / p
        r[1] += kx
        r[3] += ky
    elif name == "RFCavityPass":
        slip = round(e.Frequency * period) / e.Frequency - period
        phase = 2.0 * math.pi * e.Frequency * ((r[5] - e.TimeLag) / C_LIGHT - slip * turn)
        r[4] -= e.Voltage / gamma[1] * np.sin(phase)
    elif name == "ThinMPolePass":
        re, im = _field(r, e)
        r[1] -= re
        r[3] += im
    elif name in _THICK:
        bend, radiates = _THICK[name]
        rad = _RADIATION * gamma[0] ** 3 if radiates else 0.0
        h = e.BendingAngle / e.Length if bend else 0.0
        if bend:
            t = h * math.tan(e.EntranceAngle)
            r[1] += t * r[0]
            r[3] -= t * r[2]
        step = e.Length / e.NumIntSteps
        drifts, kicks = _slices()
        for _ in range(e.NumIntSteps):
            for d, k in zip(drifts, kicks):
                _drift(r, d * step)
                _kick(r, e, k * step, h, rad)
            _drift(r, drifts[3] * step)
        if bend:
            t = h * math.tan(e.ExitAngle)
            r[1] += t * r[0]
            r[3] -= t * r[2]
    else:
        raise NotImplementedError(name)


_THICK = {"StrMPoleSymplectic4Pass": (False, False), "BndMPoleSymplectic4Pass": (True, False),
          "StrMPoleSymplectic4RadPass": (False, True), "BndMPoleSymplectic4RadPass": (True, True)}
# 2 r_e / 3: relative energy radiated per gamma^3, curvature squared and length
_RADIATION = 2.0 / 3.0 * 2.8179403205e-15


def _gamma(ring):
    return ring.energy / ring.particle.rest_energy, ring.energy


def _exact_track(ring, beam, turns, every=False):
    """(final (6, n), coordinates at the loss (6, n), copies before every element
    and at the end of each turn, or at each turn's end)."""
    r = np.array(beam, dtype=np.float64)
    n = r.shape[1]
    coord = np.zeros((6, n))
    alive = np.ones(n, bool)
    gamma = _gamma(ring)
    period = sum(getattr(e, "Length", 0.0) for e in ring) / C_LIGHT
    copies = []
    with np.errstate(all="ignore"):
        for t in range(turns):
            for e in ring:
                if every:
                    copies.append(r.copy())
                if alive.all():
                    _element(r, e, gamma, period, t)
                else:
                    part = r[:, alive]
                    _element(part, e, gamma, period, t)
                    r[:, alive] = part
                gone = alive & ~(np.all(np.abs(r[:5]) <= 1.0, axis=0) & np.isfinite(r[5]))
                if gone.any():
                    coord[:, gone] = r[:, gone]
                    r[:, gone] = 0.0
                    r[0, gone] = np.nan
                    alive &= ~gone
            if every:
                copies.append(r.copy())
    return r, coord, copies


def exact(case, seed):
    kind = case["kind"]
    if kind in ("aperture", "serve", "gradient"):
        return None  # many turns, or a reverse pass, of 2,241 elements
    ring = _ring(case, seed)
    if kind == "optics":
        return _exact_optics(ring)
    if kind == "envelope":
        return {"mats": _exact_element_matrices(ring, _orbits(len(ring), seed)), "diff": None}
    n, t = case["n"], case["turns"]
    small = case.get("ring") == "fodo"
    if t > (8 if small else 4) or n * t > (40000 if small else 4000):
        return None
    every = kind == "monitors" or bool(case.get("refpts"))
    r, coord, copies = _exact_track(ring, _beam(case, seed), t, every)
    if kind == "host":
        out = np.asfortranarray(np.stack(copies, axis=2))[..., None] if every else None
        loss = {"islost": None, "turn": None, "elem": None, "coord": coord}
        return {"r": r, "copies": out, "loss": loss}
    if kind == "first":
        return {"r": r, "coord": coord.T.copy()}
    r = r if case.get("soa") else r.T.copy()
    if kind == "monitors":
        return {"r": r, "copies": np.stack([c.T for c in copies])[None]}
    return {"r": r, "coord": coord.T.copy()}


def _exact_element_matrices(ring, orbits):
    gamma = _gamma(ring)
    d = 0.5 * MATRIX_STEP * np.eye(6)
    mats = np.empty((len(ring), 6, 6))
    for i, e in enumerate(ring):
        r = orbits[:, i:i + 1] + np.concatenate([d, -d], axis=1)
        _element(r, e, gamma, 0.0, 0)
        mats[i] = (r[:, :6] - r[:, 6:]) / MATRIX_STEP
    return mats


def _exact_optics(ring):
    step = physics.DConstant.XYStep
    d = np.concatenate([np.zeros((6, 1)), 0.5 * step * np.eye(6, 4), -0.5 * step * np.eye(6, 4)], 1)
    x = np.zeros(6)
    for _ in range(6):
        r, _, _ = _exact_track(ring, x[:, None] + d, 1)
        m = (r[:4, 1:5] - r[:4, 5:]) / step
        x[:4] -= np.linalg.solve(m - np.eye(4), r[:4, 0] - x[:4])
    r, _, copies = _exact_track(ring, x[:, None] + d, 1, True)
    copies = np.stack(copies)
    return {"orbit": x, "orbits": copies[:, :, 0],
            "m44": (r[:4, 1:5] - r[:4, 5:]) / step,
            "mats": (copies[:, :4, 1:5] - copies[:, :4, 5:]) / step}
