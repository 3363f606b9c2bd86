"""A tape whose pool runs out: the pool's counter stops, and the photons left without are replayed."""

import time

import numpy as np
import pytest

from test_gpu_tape import _both, _run
from toys import sphere_toy

pytestmark = pytest.mark.gpu

KEY = ("surfaces/Wall/REFLECTIVITY",)


def _sphere(facets, n):
    """A bright sphere of some 460 vertices a photon (with facets half of its reflections are facet paths)."""
    extra = dict(p_spike=0.0, p_lobe=0.5, p_back=0.0, sigma_alpha=0.2)
    det = sphere_toy(1.0, "UNIFIED_METAL" if facets else "PAINTED", R=0.99, L_abs=1e3, extra=extra if facets else None)
    return _run(det, KEY, (0.1, 0.0, 0.0), 400.0, (n,))


def _pool(tape, n):
    """The pool's chunks: the tape less its control cells, first chunks and replay list."""
    return (tape.numel() // 16 - 4 - 4 * n - (n + 4) // 4) // 16


@pytest.mark.parametrize("facets", [False, True])
def test_the_pools_counter_stops(gpu, facets):
    """Each wavefront asks an empty pool once: a counter that grew with every photon would wrap at 2^26 of them, and
    chunks would be handed out twice."""
    import torch

    n = 1 << 20
    run = _sphere(facets, n)
    a, b, tape = _both(run)
    asked, pool = int(tape[:4].view(torch.int32).item()), _pool(tape, n)
    waves = 12 * run.eng.last_launch()["grid"]
    assert pool < asked <= pool + 64 * waves
    assert np.linalg.norm(b - a) <= 2e-6 * np.linalg.norm(a)


def _ms(run, tape):
    """The adjoint's time, the best of three after a first."""
    import torch

    out = []
    for _ in range(4):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        run._launch_adjoint(tape=tape)
        torch.cuda.synchronize()
        out.append(1e3 * (time.perf_counter() - t0))
    return min(out[1:])


@pytest.mark.parametrize("n", [1 << 20, 1 << 22])
def test_an_empty_pool_costs_little(gpu, n):
    """Most photons find no room: the adjoint's own walk ends them there (a walk to their end, then the two of the
    replay, took 1.4 times the replay), and the replay evens them out over the wavefronts (equal shares of 2^22 took
    another 1.4).  A quarter is room for the taped share's walk and the clocks."""
    run = _sphere(True, n)
    a, b, tape = _both(run)
    assert np.linalg.norm(b - a) <= 2e-6 * np.linalg.norm(a)
    assert _ms(run, tape) <= 1.25 * _ms(run, None)


@pytest.mark.parametrize("n,chunk", [(100_001, 100), (1 << 18, 64), (1 << 21, 0), ((1 << 18) + 63, 2048)])
def test_every_photon_left_is_replayed_once(gpu, n, chunk):
    """The replay of a list in first ranges alone, with the work queue's chunks, and in chunks that a few wavefronts
    take all of."""
    from lumen_amd import _lib
    from lumen_amd.api import Controls

    run = _sphere(True, n)
    a, _, tape = _both(run)
    run.grad.zero_()
    run.adj_health.zero_()
    run._launch_adjoint(Controls(chunk=chunk), tape=tape)
    b = run.grad.cpu().numpy()
    assert float(run.adj_health.cpu()[_lib.HEALTH_NAMES.index("photons")]) == n
    assert np.linalg.norm(b - a) <= 2e-6 * np.linalg.norm(a)
