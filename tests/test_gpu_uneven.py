"""Sources of unequal path lengths in one launch: however they lie, the engine's own split of the photons over the
wavefronts is no slower than a queue of 256-photon chunks, which leaves no wavefront more than that."""

import time

import numpy as np
import pytest

from lumen_amd.api import Controls
from lumen_amd.batch import BatchRun
from lumen_amd.sources import Batch, Point
from toys import sphere_toy

pytestmark = pytest.mark.gpu

N = 1 << 22
KEYS = ("surfaces/Wall/REFLECTIVITY",)


def _run(where):
    """64 sources in a bright sphere, of which eight have some 270 vertices a photon and the others 1: 300 nm is shifted
    at once, with a yield that leaves nothing."""
    det = sphere_toy(1.0, "PAINTED", R=0.98, L_abs=1e3, L_wls=0.01, wls_yield=1e-4)
    long = {"first": lambda i: i < 8, "every eighth": lambda i: i % 8 == 0}[where]
    srcs = tuple(Point((0.1, 0.05, -0.02), lam=500.0 if long(i) else 300.0, n_photons=1e5) for i in range(64))
    return BatchRun(det, Batch(srcs, (N // 64,) * 64), seed=3, grad_keys=KEYS, tune=False, graph=False)


def _ms(fn):
    import torch

    out = []
    for _ in range(4):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        fn()
        torch.cuda.synchronize()
        out.append(1e3 * (time.perf_counter() - t0))
    return min(out[1:])


@pytest.mark.parametrize("what", ["forward", "adjoint"])
@pytest.mark.parametrize("where", ["first", "every eighth"])
def test_long_paths_side_by_side(gpu, where, what):
    run = _run(where)
    res = []
    for ctl in (Controls(), Controls(chunk=256)):
        if what == "forward":
            ms = _ms(lambda: run._fwd_body(ctl))  # noqa: B023
            res.append((ms, run.tally.cpu().numpy().copy()))
        else:
            run.cot.fill_(1.0)
            ms = _ms(lambda: run._launch_adjoint(ctl))  # noqa: B023
            run.grad.zero_()
            run._launch_adjoint(ctl)
            res.append((ms, run.grad.cpu().numpy().copy()))
    (own, a), (chunks, b) = res
    # the same deposits (terms) in FP64 sums of another order: n roundings of 1.1e-16 at most
    np.testing.assert_allclose(a, b, rtol=N * 1.2e-16, atol=N * 1.2e-16 * np.abs(b).max())
    assert own <= 1.25 * chunks


WAVES = 256 * 12  # wavefronts of a launch on 256 CUs
OWN = 256 * WAVES  # the photons that wavefronts have of their own; past them 8 parts of the queue, chunks of 64


@pytest.mark.parametrize("n,chunk", [(64 * WAVES, 0), (64 * WAVES + 1, 0), (OWN - 1, 0), (OWN, 0), (OWN + 1, 0),
                                     (OWN + 64, 0), (OWN + 8 * 64, 0), (OWN + 8 * 64 + 1, 0), (OWN + 33 * 64 + 5, 0),
                                     (5000, 1), (WAVES * 7 + 1, 7), (WAVES * 7 + 8 * 7 + 1, 7), (100_003, 1 << 17)])
def test_every_photon_once_at_the_edges_of_the_split(gpu, n, chunk):
    """The last own block, the queue's first chunk, a part that is one chunk short, chunks of 1 and of more than all."""
    import lumen_amd as L
    from lumen_amd.detector import example_tank

    det = example_tank()
    src = L.sources.Point((0.05, 0.0, 0.1), lam=400.0, n_photons=2e5)
    a = L.simulate(det, src, samples=n, seed=4, controls=Controls(chunk=chunk))
    b = L.simulate(det, src, samples=n, seed=4, chunk=50_000)  # launches of photons that are all own
    for k in ("photons", "vertices", "records"):
        assert getattr(a.health, k) == getattr(b.health, k)
    assert a.health.photons == n
    # the same deposits in FP64 sums of another order: n roundings of 1.1e-16 at most
    for x, y in ((a.arrivals, b.arrivals), (a.charge, b.charge), (a.arrival2, b.arrival2)):
        np.testing.assert_allclose(x.cpu().numpy(), y.cpu().numpy(), rtol=n * 1.2e-16, atol=0.0)
