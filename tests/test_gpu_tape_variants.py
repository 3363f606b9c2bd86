"""The adjoint from a tape against the replay of the same photons, in the kernels and options the plain runs leave out:
shifted wavelengths with facets, BVH nodes in memory, tables that do not fit the reader's LDS, sensors credited with the
volume left, every charge cell, other controls, a backward run twice; and the replay's own schedule, on launches that
take no tape.

Both add the same float32 terms in FP64 in another order; a term is some ten roundings of 2^-24 where a kernel contracts
another product than the other, and no photon of these seeds sits on an edge: 2e-6 of the gradient's norm.
"""

import numpy as np
import pytest

import lumen_amd as L
from lumen_amd import _lib
from lumen_amd.api import Controls, engine
from lumen_amd.batch import BatchRun
from lumen_amd.detector import example_tank, lar_box, water_tank
from lumen_amd.params import Table
from lumen_amd.sources import Batch, Point
from toys import sensor_volume_toy, sphere_toy

pytestmark = pytest.mark.gpu

WALL = "surfaces/Wall/"
FACETS = dict(p_spike=0.0, p_lobe=0.5, p_back=0.0, sigma_alpha=0.2)
KNOTS = np.linspace(1.5, 5.0, 8000)  # as many gradient slots as a block's LDS holds beside the reader's lists

# name: (detector, keys, wavelength, photons)
DETS = {
    "plain": (lambda: sphere_toy(1.0, "PAINTED", R=0.9, L_ray=3.0), (WALL + "REFLECTIVITY",
              "materials/Water/ABSLENGTH", "materials/Water/RAYLEIGH"), 400.0, 20000),
    "wls": (lambda: sphere_toy(1.0, "PAINTED", R=0.9, L_wls=1.0), (WALL + "REFLECTIVITY",
            "materials/Water/WLSABSLENGTH"), 300.0, 20000),
    "wls with facets": (lambda: sphere_toy(1.0, "UNIFIED_METAL", R=0.9, L_wls=1.0, extra=FACETS),
                        (WALL + "REFLECTIVITY", WALL + "sigma_alpha", "materials/Water/WLSABSLENGTH"), 300.0, 20000),
    "argon": (lar_box, ("materials/LAr/RAYLEIGH", "surfaces/PTFE/REFLECTIVITY"), 128.0, 1000),
    "tank": (water_tank, ("materials/Water/ABSLENGTH", "surfaces/Liner/sigma_alpha"), 410.0, 20000),
    "cells": (example_tank, ("materials/Water/ABSLENGTH",), 400.0, 20000),
    "exit": (lambda: sensor_volume_toy("exit", keyed=True, L_abs=5.0),
             ("surfaces/sensor/EFFICIENCY", "materials/Water/ABSLENGTH"), 400.0, 20000),
    "many slots": (lambda: sphere_toy(1.0, "PAINTED", R=0.9, extra=dict(eff=Table(KNOTS, 0.5 + 0.05 * KNOTS))),
                   (WALL + "eff",), 400.0, 20000),
    "many slots, wls with facets": (lambda: sphere_toy(1.0, "UNIFIED_METAL", R=0.9, L_wls=1.0, extra=dict(
        FACETS, sigma_alpha=Table(KNOTS[::2], 0.1 + 0.02 * KNOTS[::2]))), (WALL + "sigma_alpha",), 300.0, 20000),
}


def _same(name, controls):
    import torch

    mk, keys, lam, n = DETS[name]
    src = Batch((Point((0.03, 0.02, -0.01), lam=lam, n_photons=1e5), Point((0.0, 0.1, 0.05), lam=lam, n_photons=1e5)),
                (n, n // 3))
    run = BatchRun(mk(), src, seed=5, grad_keys=keys, tune=False, graph=False, controls=controls)
    ctl = controls.struct()
    forward = run.eng.tape(ctl, False, run.total, False)
    tape = forward if forward is not None else run.eng.tape(ctl, False, run.total, True)
    assert tape is not None
    tape.fill_(0xAB)  # nothing is read that was not written
    run._fwd_body(tape=forward)
    feat = run.eng.last_launch()["features"]
    S, K = run.eng.S, run.eng.K
    run.cot.zero_()
    run.cot[:, :S] = 0.1
    run.cot[:, 3 * S:3 * S + S * K] = torch.linspace(0.5, 1.5, S * K, dtype=torch.float64, device="cuda")
    out = []
    for t in (None, tape):
        run.grad.zero_()
        run.adj_health.zero_()
        run._launch_adjoint(tape=t)
        out.append(run.grad.cpu().numpy().copy())
    assert float(run.adj_health.cpu()[_lib.HEALTH_NAMES.index("photons")]) == run.total
    assert np.linalg.norm(out[0]) > 0.0
    assert np.linalg.norm(out[1] - out[0]) <= 2e-6 * np.linalg.norm(out[0])
    return feat


@pytest.mark.parametrize("name", sorted(DETS))
def test_the_tape_is_the_replay(gpu, name):
    _same(name, Controls())


@pytest.mark.parametrize("name", ["plain", "wls with facets", "argon", "tank"])
def test_with_nodes_in_memory(gpu, name):
    feat = _same(name, Controls(nodes_global=True))
    assert feat & 8


OTHER = [Controls(roulette=0.4), Controls(max_vertices=3), Controls(keep_zero_weight=True),
         Controls(chunk=64, tally_global=True)]


@pytest.mark.parametrize("name,controls", [(n, c) for n in ("plain", "wls with facets", "tank") for c in OTHER]
                         + [(n, Controls(max_distance=0.7)) for n in ("plain", "wls with facets")])
def test_with_other_controls(gpu, name, controls):
    _same(name, controls)


@pytest.mark.parametrize("name", ["cells", "wls", "tank"])
def test_a_backward_run_twice(gpu, name):
    import torch

    from lumen_amd.autograd import simulate_diff, table_tensor

    mk, keys, lam, n = DETS[name]
    det = mk()
    t = table_tensor(det.params(), keys[0])
    light = simulate_diff(det, Point((0.03, 0.02, -0.01), lam=lam, n_photons=1e5), {keys[0]: t}, samples=n, seed=5)
    a, b = light.arrivals.sum(), (light.arrivals * 2.0).sum()
    first, = torch.autograd.grad(a, t, retain_graph=True)
    twice, = torch.autograd.grad(b, t, retain_graph=True)
    again, = torch.autograd.grad(a, t)
    # doubled exactly but for the order of the FP64 sums; the gradient is rounded to float32 once
    np.testing.assert_allclose(twice.cpu().numpy(), 2.0 * first.cpu().numpy(), rtol=2.5e-7, atol=0.0)
    np.testing.assert_allclose(again.cpu().numpy(), first.cpu().numpy(), rtol=2.5e-7, atol=0.0)


WAVES = 256 * 12  # wavefronts of a launch on 256 CUs


@pytest.mark.parametrize("n", [1, 63, 65, WAVES - 1, WAVES + 1, 384 * WAVES, 384 * WAVES + 1, 1536 * WAVES + 321])
def test_every_photon_once_in_the_replay(gpu, n):
    """Separate reference values: no tape, so the adjoint's kernel hands out the photons by its own split."""
    import torch

    from lumen_amd.autograd import simulate_diff

    det = example_tank()
    key = "materials/Water/ABSLENGTH"
    src = L.sources.Point((0.05, 0.0, 0.1), lam=400.0, n_photons=2e5)
    assert all(engine(det).tape(Controls().struct(), True, n, by) is None for by in (False, True))
    grads = []
    for ctl in (None, Controls(chunk=100)):
        t = torch.tensor(np.asarray(det.params().flat()[key]), dtype=torch.float64, device="cuda", requires_grad=True)
        light = simulate_diff(det, src, {key: t}, samples=n, seed=4, controls=ctl, reference=det.params())
        light.arrivals.sum().backward()
        run = light.provenance["run"]
        assert float(run.adj_health.cpu()[_lib.HEALTH_NAMES.index("photons")]) == n
        grads.append(t.grad.cpu().numpy())
    # the packed gradient is rounded to float32 once
    np.testing.assert_allclose(grads[0], grads[1], rtol=2.5e-7, atol=0.0)
