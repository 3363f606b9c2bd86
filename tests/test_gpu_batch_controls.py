"""A staged run whose controls are replaced between calls: the tape of its adjoint follows them."""

import numpy as np
import pytest

from lumen_amd.api import Controls
from lumen_amd.batch import BatchRun
from lumen_amd.detector import lar_box, water_tank
from lumen_amd.sources import Batch, Point

pytestmark = pytest.mark.gpu

DETS = {"tank": (water_tank, ("materials/Water/ABSLENGTH", "surfaces/Liner/REFLECTIVITY"), 410.0, 3000),
        "lar": (lar_box, ("surfaces/PTFE/REFLECTIVITY",), 128.0, 200)}  # the adjoint's own walk, the forward's tape


def _run(where, controls=None):
    mk, keys, lam, n = DETS[where]
    batch = Batch(tuple(Point(p, lam=lam, n_photons=float(n)) for p in ((0.3, 0.2, -0.1), (0.0, 0.1, 0.4))), (n, n + 1))
    return BatchRun(mk(), batch, seed=3, grad_keys=keys, tune=False, graph=False, controls=controls)


def _loss(run):
    import torch

    S = run.eng.S
    cot = torch.zeros_like(run.tally)
    cot[:, 3 * S:4 * S] = torch.linspace(0.5, 1.5, S, dtype=torch.float64, device="cuda")
    return lambda tally: cot


# controls that take no tape, that trace other paths, and that launch the same ones another way
@pytest.mark.parametrize("then", [Controls(reach_bound=True), Controls(jump=True), Controls(max_vertices=2),
                                  Controls(roulette=0.3), Controls(chunk=64, nodes_global=True)])
@pytest.mark.parametrize("where", sorted(DETS))
def test_controls_replaced_after_a_first_call(gpu, where, then):
    run = _run(where)
    loss = _loss(run)
    run.forward_adjoint(loss)
    if then.jump:
        run.eng.ensure_jump()
    run.controls = then
    got = run.forward_adjoint(loss).cpu().numpy().copy()
    # the trace at the new controls, the adjoint at the run's own
    ref = _run(where)
    ref.controls = then
    ref._fwd_body()
    ref.cot.copy_(loss(ref.tally))
    ref.grad.zero_()
    ref.adj_health.zero_()
    ref._launch_adjoint(Controls())
    want = ref.grad.cpu().numpy()
    assert np.linalg.norm(want) > 0.0
    # the same float32 terms added in FP64, a term some ten roundings of 2^-24 where a kernel contracts another product
    assert np.linalg.norm(got - want) <= 2e-6 * np.linalg.norm(want)
    run.controls = Controls()
    back = run.forward_adjoint(loss).cpu().numpy()
    assert np.linalg.norm(back - _run(where).forward_adjoint(loss).cpu().numpy()) <= 2e-6 * np.linalg.norm(back)


def test_an_eager_call_between_replays(gpu):
    """A graph that was captured with one tape is captured again once another was taken."""
    run = _run("tank")
    run.graph = True
    loss = _loss(run)
    a = run.forward_adjoint(loss).cpu().numpy().copy()
    run.graph = False
    run.controls = Controls(reach_bound=True)
    run.forward_adjoint(loss)
    run.controls = Controls()
    run.graph = True
    for _ in range(2):
        b = run.forward_adjoint(loss).cpu().numpy()
        assert np.linalg.norm(b - a) <= 2e-6 * np.linalg.norm(a)


@pytest.mark.parametrize("where", sorted(DETS))
def test_the_adjoint_of_a_tape_has_the_forwards_launch_shape(gpu, where, monkeypatch):
    from lumen_amd import batch

    monkeypatch.setattr(batch, "tuned_controls", lambda run, what: Controls(chunk=192))
    mk, keys, lam, n = DETS[where]
    src = Batch((Point((0.3, 0.2, -0.1), lam=lam, n_photons=float(n)),), (n,))
    tuned = BatchRun(mk(), src, seed=3, grad_keys=keys, graph=False)
    plain = BatchRun(mk(), src, seed=3, grad_keys=keys, graph=False, tune=False)
    a, b = (r.forward_adjoint(_loss(r)).cpu().numpy() for r in (tuned, plain))
    assert tuned._tape is not None and tuned.adj_controls.chunk == tuned.controls.chunk == 192
    assert np.linalg.norm(a - b) <= 2e-6 * np.linalg.norm(b)
