"""How a launch's photons are handed out to its wavefronts: at every edge of the split (fewer photons than wavefronts,
one more than they hold at once, the work queue's first and last chunks) each photon is traced once, forward and
adjoint, against the same photons in explicit chunks."""

import numpy as np
import pytest

import lumen_amd as L
from lumen_amd.api import Controls, engine
from lumen_amd.detector import example_tank

pytestmark = pytest.mark.gpu

SRC = L.sources.Point((0.05, 0.0, 0.1), lam=400.0, n_photons=2e5)
WAVES = 256 * 12  # wavefronts of a launch on 256 CUs
SIZES = [1, 63, 64, 65, 255, 256, 257, WAVES - 1, WAVES, WAVES + 1, 2 * WAVES + 1, 384 * WAVES, 384 * WAVES + 1,
         1536 * WAVES + 64 * 5 + 1]


@pytest.fixture(scope="module")
def det(gpu):
    return example_tank()


@pytest.mark.parametrize("n", SIZES)
def test_every_photon_once(det, n):
    a = L.simulate(det, SRC, samples=n, seed=4)
    b = L.simulate(det, SRC, samples=n, seed=4, controls=Controls(chunk=100))
    assert engine(det).last_launch()["grid"] > 0
    for k in ("photons", "vertices", "records"):
        assert getattr(a.health, k) == getattr(b.health, k)
    assert a.health.photons == n
    # the same deposits in FP64 sums of another order: n roundings of 1.1e-16 at most
    for x, y in ((a.arrivals, b.arrivals), (a.charge, b.charge), (a.arrival2, b.arrival2)):
        np.testing.assert_allclose(x.cpu().numpy(), y.cpu().numpy(), rtol=max(n, 16) * 1.2e-16, atol=0.0)


@pytest.mark.parametrize("n", [1, 65, WAVES + 1, 384 * WAVES + 1])
def test_every_photon_once_in_the_adjoint(det, n):
    import torch

    from lumen_amd.autograd import simulate_diff

    key = "materials/Water/ABSLENGTH"
    flat = det.params().flat()[key]
    grads = []
    for ctl in (None, Controls(chunk=100)):
        t = torch.tensor(np.asarray(flat), dtype=torch.float64, device="cuda", requires_grad=True)
        light = simulate_diff(det, SRC, {key: t}, samples=n, seed=4, controls=ctl)
        light.arrivals.sum().backward()
        run = light.provenance["run"]
        assert float(run.adj_health.cpu()[13]) == n
        grads.append(t.grad.cpu().numpy())
    # the packed gradient is rounded to float32 once
    np.testing.assert_allclose(grads[0], grads[1], rtol=2.5e-7, atol=0.0)
