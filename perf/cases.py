"""The timed work of this framework: what its users have it do, through its public entry points.

    listed()             the named cases, smallest calls to largest
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  what a program holds before the call (detector, sources, values, target), made from the seed
    run(state)           one pass, and its whole outputs
    work(case)           the bytes and FP32 operations a pass cannot do without
    exact(case, seed)    None: see there

Four kinds of program are here.  A forward simulation (``simulate``) gives each sensor's light: the tutorial's 8-PMT
cube, an event in the 1,000-PMT water tank, the same with the time histogram, or with its random choices drawn at
reference values (the common-random-number run of a systematic or a finite difference).  A fit's step
(``simulate_diff`` and a backward through it) adds the gradient of a Poisson likelihood.  A batch of many uneven
sources (a calibration scan) goes through ``simulate(det, Batch(...))`` once, or through a staged ``BatchRun`` that a
fit replays.  The liquid-argon box is the long-path workload: 150 to 280 vertices a photon, against 1 to 2 in water.
"""

from __future__ import annotations

import math
import random

import numpy as np
import torch

import lumen_amd as L
from lumen_amd.autograd import simulate_diff
from lumen_amd.batch import BatchRun
from lumen_amd.detector import example_tank, lar_box, water_tank
from lumen_amd.sources import Batch, CherenkovSegment, Point

TANK_KEYS = ("materials/Water/ABSLENGTH", "materials/Water/RAYLEIGH", "surfaces/Liner/REFLECTIVITY",
             "surfaces/Liner/sigma_alpha")
LAR_KEYS = ("materials/LAr/RAYLEIGH", "surfaces/PTFE/REFLECTIVITY")
QE = 0.25

# FP32 operations of the photon loop's algorithm per photon (add, sub, mul, div, compare, math function = 1), counted
# by the op-counting walk of the tests' oracle: the tutorial's point source, the tank's Cherenkov track and point
# sources, and the mean over positions of the LAr box
OPS = {"example": 564.0, "tank": 3170.0, "lar": 130000.0}
SENSORS = {"example": 8, "tank": 1000, "lar": 120}
CHARGE = {"example": 2, "tank": 1, "lar": 1}  # at least so many charge cells a sensor
GATE_NODES = 41


def listed():
    return [
        # the tutorial's detector with a quick preview's photons: the smallest call, launches and latency
        dict(name="tutorial_preview", kind="tutorial", photons=1 << 12, lam=400.0),
        # the tutorial itself: 2^18 photons of a 400 nm point source
        dict(name="tutorial", kind="tutorial", photons=1 << 18, lam=400.0),
        # one event of a reconstruction's scan over hypotheses: a track with an odd, modest photon count
        dict(name="tank_event", kind="event", photons=100003, length=1.0),
        # the headline: the 1 m track at 2^24 photons
        dict(name="tank_event_full", kind="event", photons=1 << 24, length=1.0),
        # an event with its time histogram over a 40 ns gate (what a waveform is built from)
        dict(name="tank_timing", kind="timing", photons=1 << 20, length=0.6),
        # a systematic's shifted light at common random numbers: values moved, choices drawn at the reference's
        dict(name="tank_shift", kind="shift", photons=1 << 21, shift=1.001),
        # an optimiser's step on few photons: forward and backward, the host's share visible
        dict(name="tank_fit_step", kind="fit", photons=131071, length=1.0),
        # the calibration gradient at full statistics
        dict(name="tank_fit_full", kind="fit", photons=1 << 23, length=1.0),
        # a scan of many uneven point sources as one call
        dict(name="tank_batch", kind="batch", sources=64, lo=10, hi=16, counts=6),
        # the 256-source calibration batch, replayed by a fit: forward, the sources' likelihoods, backward
        dict(name="tank_batch_fit", kind="batch_fit", sources=256, lo=12, hi=20, counts=6),
        # a light map of the liquid-argon box: a voxel grid of VUV sources, forward
        dict(name="lar_map", kind="lar_map", side=8, photons=4096),
        # the argon box's calibration step: forward and backward over a coarser grid
        dict(name="lar_fit", kind="lar_fit", side=4, photons=4096),
    ]


def draw(rng: random.Random):
    def log2(lo, hi):
        return int(2.0 ** rng.uniform(lo, hi))

    kind = rng.choice(("tutorial", "event", "timing", "shift", "fit", "batch", "batch_fit", "lar_map", "lar_fit"))
    if kind == "tutorial":
        return dict(kind=kind, photons=log2(12, 20), lam=round(rng.uniform(350.0, 500.0), 1))
    if kind == "event":
        return dict(kind=kind, photons=log2(12, 24), length=round(rng.uniform(0.2, 1.5), 2))
    if kind == "timing":
        return dict(kind=kind, photons=log2(14, 22), length=round(rng.uniform(0.2, 1.5), 2))
    if kind == "shift":
        return dict(kind=kind, photons=log2(14, 22), shift=round(rng.uniform(0.95, 1.05), 3))
    if kind == "fit":
        return dict(kind=kind, photons=log2(14, 23), length=round(rng.uniform(0.2, 1.5), 2))
    if kind == "batch":
        return dict(kind=kind, sources=rng.randint(8, 128), lo=10, hi=rng.randint(12, 16), counts=rng.randint(0, 999))
    if kind == "batch_fit":
        return dict(kind=kind, sources=rng.randint(16, 256), lo=12, hi=rng.randint(14, 19), counts=rng.randint(0, 999))
    if kind == "lar_map":
        return dict(kind=kind, side=rng.randint(3, 8), photons=log2(8, 12))
    return dict(kind=kind, side=rng.randint(2, 4), photons=log2(9, 12))


_DETECTORS = {}


def _detector(name):
    """A program builds its detector once and keeps it."""
    if name not in _DETECTORS:
        _DETECTORS[name] = {"example": example_tank, "tank": water_tank, "lar": lar_box}[name]()
    return _DETECTORS[name]


def _where(case):
    kind = case["kind"]
    return "example" if kind == "tutorial" else "lar" if kind.startswith("lar") else "tank"


def _track(rng, length):
    """A track of ``length`` m inside the tank's fiducial cylinder (R 1.8 m, half height 1.3 m)."""
    while True:
        r, ph, z = 1.8 * math.sqrt(rng.uniform()), rng.uniform(0, 2 * math.pi), rng.uniform(-1.3, 1.3)
        x0 = np.array([r * math.cos(ph), r * math.sin(ph), z])
        d = rng.normal(size=3)
        d /= np.linalg.norm(d)
        x1 = x0 + length * d
        if math.hypot(x1[0], x1[1]) < 1.8 and abs(x1[2]) < 1.3:
            return CherenkovSegment("Water", start=tuple(map(float, x0)), direction=tuple(map(float, d)),
                                    length=float(length))


def _counts(case):
    """The batch's photon counts: uneven, 2^U with U uniform on [lo, hi]; a part of the case, not of the seed."""
    u = np.random.default_rng(case["counts"]).uniform(case["lo"], case["hi"], case["sources"])
    return [int(n) for n in np.round(2.0**u)]


def _tank_batch(case, rng):
    """Isotropic monochromatic points (350-500 nm) uniform in the fiducial cylinder."""
    counts = _counts(case)
    srcs = []
    for n in counts:
        r, ph, z = 1.8 * math.sqrt(rng.uniform()), rng.uniform(0, 2 * math.pi), rng.uniform(-1.3, 1.3)
        srcs.append(Point((r * math.cos(ph), r * math.sin(ph), z), lam=float(rng.uniform(350.0, 500.0)),
                          n_photons=float(n)))
    return Batch(tuple(srcs), tuple(counts))


def _voxels(case, rng):
    """128 nm points at the centres of a side^3 voxel grid of the argon box, the grid moved by the seed."""
    n, half = case["side"], (2.5, 2.0, 2.5)
    axes = [(-h + (np.arange(n) + 0.5 + rng.uniform(-0.3, 0.3)) * (2 * h / n)) for h in half]
    pts = [Point((float(x), float(y), float(z)), lam=128.0, n_photons=float(case["photons"]))
           for x in axes[0] for y in axes[1] for z in axes[2]]
    return Batch(tuple(pts), (int(case["photons"]),) * len(pts))


def _poisson(S, target):
    """loss(tally) -> dLoss/dtally of the per-source Poisson likelihood sum_s pe - target log pe, pe = QE charge."""

    def loss(tally):
        pe = QE * tally[:, 3 * S:4 * S]
        cot = torch.zeros_like(tally)
        cot[:, 3 * S:4 * S] = QE * (1.0 - target / torch.clamp(pe, min=1e-30))
        return cot

    return loss


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    det = _detector(_where(case))
    s = dict(kind=kind, det=det, seed=int(seed))
    if kind == "tutorial":
        s["source"] = Point(tuple(float(v) for v in rng.uniform(-0.2, 0.2, 3)), lam=case["lam"], n_photons=2e5)
        s["n"], s["params"] = case["photons"], det.params()
    elif kind in ("event", "timing"):
        s["source"], s["n"], s["params"] = _track(rng, case["length"]), case["photons"], det.params()
    elif kind == "shift":
        s["source"], s["n"], s["reference"] = _track(rng, 1.0), case["photons"], det.params()
        s["params"] = det.params().scale("materials/Water/ABSLENGTH", case["shift"])
    elif kind == "fit":
        s["source"], s["n"], p = _track(rng, case["length"]), case["photons"], det.params()
        true = p.scale("materials/Water/ABSLENGTH", 1.05).scale("surfaces/Liner/REFLECTIVITY", 0.95)
        light = L.simulate(det, s["source"], true, samples=s["n"], seed=s["seed"] + 1)
        s["target"] = L.readout.pe(light, true, det)
        s["params"] = p
        flat = p.flat()
        s["values"] = {k: torch.tensor(flat[k], dtype=torch.float32, device="cuda", requires_grad=True)
                       for k in TANK_KEYS}
    elif kind == "batch":
        s["source"], s["params"] = _tank_batch(case, rng), det.params()
    else:
        batch = _tank_batch(case, rng) if kind == "batch_fit" else _voxels(case, rng)
        fit = kind.endswith("fit")
        keys = () if not fit else LAR_KEYS if kind == "lar_fit" else TANK_KEYS
        s["run"] = run = BatchRun(det, batch, seed=s["seed"], grad_keys=keys, tune=False)
        if fit:
            S = run.eng.S
            s["loss"] = _poisson(S, 1.05 * QE * run.forward()[:, 3 * S:4 * S].clone())
    return s


def _light(light):
    return dict(arrivals=light.arrivals, error=light.arrivals_error, mean_time=light.mean_arrival_time,
                charge=light.charge)


def run(s):
    kind, det = s["kind"], s["det"]
    if kind in ("tutorial", "event", "batch"):
        light = L.simulate(det, s["source"], s["params"], samples=s.get("n"), seed=s["seed"])
        return dict(_light(light), pe=L.readout.pe(light, s["params"], det))
    if kind == "timing":
        light = L.simulate(det, s["source"], s["params"], samples=s["n"], seed=s["seed"],
                           gate=(0.0, float(GATE_NODES - 1)))
        return dict(_light(light), time=light.time, late=light.late, early=light.early)
    if kind == "shift":
        light = L.simulate(det, s["source"], s["params"], samples=s["n"], seed=s["seed"], reference=s["reference"])
        return dict(_light(light), pe=L.readout.pe(light, s["params"], det))
    if kind == "fit":
        light = simulate_diff(det, s["source"], s["values"], samples=s["n"], seed=s["seed"], params=s["params"])
        pe = L.readout.pe(light, s["params"], det)
        loss = (pe - s["target"] * torch.log(torch.clamp(pe, min=1e-30))).sum()
        grads = torch.autograd.grad(loss, list(s["values"].values()))
        return dict(pe=pe.detach(), loss=loss.detach(), grads=list(grads))
    if kind == "lar_map":
        return s["run"].forward()
    grad = s["run"].forward_adjoint(s["loss"])  # the batch fits
    return dict(tally=s["run"].tally, grad=grad)


def _photons(case):
    if case["kind"] in ("batch", "batch_fit"):
        return sum(_counts(case))
    if case["kind"].startswith("lar"):
        return case["side"] ** 3 * case["photons"]
    return case["photons"]


def work(case):
    """One walk of every photon (two with a gradient: the light first, then the derivative of its likelihood), a
    reference's walk weighed beside the live one counted once; the tallies written once (with a gradient, read once
    as a cotangent too).  The detector's tables are a few hundred KB, the photons live in registers."""
    where, kind = _where(case), case["kind"]
    events = case["sources"] if "sources" in case else case["side"] ** 3 if "side" in case else 1
    cells = SENSORS[where] * (3 + CHARGE[where] + (GATE_NODES + 4 if kind == "timing" else 0))
    fit = kind.endswith("fit")
    return {"bytes": 8.0 * cells * events * (2 if fit else 1) + 88.0 * events + 2e5,
            "flops": OPS[where] * _photons(case) * (2 if fit else 1)}


def exact(case, seed):
    """None: an output is a Monte Carlo sum over the float32 walks of given photons (their random numbers fixed by
    seed, photon and vertex).  A 64-bit walk from the same random numbers parts from its photon's wherever a drawn
    choice or a grazed edge lies within a rounding, so the sums of such walks are other samples of the same light,
    not these outputs' values in 64 bits."""
    return None
