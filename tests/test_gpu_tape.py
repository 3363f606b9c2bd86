"""The adjoint from a tape of the photons' paths (``lh_adjoint_tape``) against the replay of the same photons
(``lh_adjoint``): every path length a tape stores another way, each writer (the forward, the adjoint's own walk), a pool
that runs out, and where a launch takes no tape.

Both add the same float32 terms in FP64 in another order; a term is some ten roundings of 2^-24 where a kernel contracts
another product than the other, and no photon of these seeds sits on an edge: 2e-6 of the gradient's norm.
"""

import numpy as np
import pytest

from lumen_amd import _lib
from lumen_amd.api import Controls, engine
from lumen_amd.batch import BatchRun
from lumen_amd.detector import lar_box, water_tank
from lumen_amd.sources import Batch, Point
from toys import sphere_toy

pytestmark = pytest.mark.gpu

TANK = ("materials/Water/ABSLENGTH", "materials/Water/RAYLEIGH", "surfaces/Liner/REFLECTIVITY",
        "surfaces/Liner/sigma_alpha")
LAR = ("materials/LAr/RAYLEIGH", "surfaces/PTFE/REFLECTIVITY")


def _both(run):
    """The gradient by the replay and from the tape, with the tape's words."""
    import torch

    S = run.eng.S
    ctl = run.controls.struct()
    forward = run.eng.tape(ctl, False, run.total, False)
    tape = forward if forward is not None else run.eng.tape(ctl, False, run.total, True)
    assert tape is not None
    tape.fill_(0xAB)  # nothing is read that was not written
    run._fwd_body(tape=forward)
    run.cot.zero_()
    run.cot[:, 3 * S:4 * S] = torch.linspace(0.5, 1.5, S, dtype=torch.float64, device="cuda")
    out = []
    for t in (None, tape):
        run.grad.zero_()
        run.adj_health.zero_()
        run._launch_adjoint(tape=t)
        out.append(run.grad.cpu().numpy().copy())
    assert float(run.adj_health.cpu()[_lib.HEALTH_NAMES.index("photons")]) == run.total
    return out[0], out[1], tape


def _run(det, keys, pos, lam, counts):
    srcs = tuple(Point(pos, lam=lam, n_photons=float(n)) for n in counts)
    return BatchRun(det, Batch(srcs, tuple(counts)), seed=3, grad_keys=keys, tune=False, graph=False)


@pytest.mark.parametrize("counts", [(1,), (64,), (65, 1, 3000), (40000,)])
@pytest.mark.parametrize("where", ["tank", "lar"])
def test_tape_equals_the_replay(gpu, where, counts):
    det, keys, lam = (water_tank(), TANK, 410.0) if where == "tank" else (lar_box(), LAR, 128.0)
    counts = tuple(max(n // 20, 1) for n in counts) if where == "lar" else counts
    a, b, _ = _both(_run(det, keys, (0.3, 0.2, -0.1), lam, counts))
    assert np.linalg.norm(b - a) <= 2e-6 * np.linalg.norm(a)


@pytest.mark.parametrize("n", [2000, 60000])
def test_long_paths_and_a_pool_that_runs_out(gpu, n):
    """A bright diffuse sphere: some 460 vertices a photon, in pool chunks of 15 records; the larger run asks for more
    chunks than the tape has, and the photons without are replayed."""
    import torch

    run = _run(sphere_toy(1.0, "PAINTED", R=0.99, L_abs=1e3), ("surfaces/Wall/REFLECTIVITY",), (0.1, 0.0, 0.0), 400.0,
               (n,))
    a, b, tape = _both(run)
    chunks = (tape.numel() - 64 * n) // 256  # at least the pool's
    asked = int(tape[:4].view(torch.int32).item())
    assert asked > chunks if n == 60000 else 0 < asked <= chunks
    assert np.linalg.norm(b - a) <= 2e-6 * np.linalg.norm(a)


def test_where_a_launch_takes_no_tape(gpu):
    eng = engine(water_tank(), "cuda")
    ctl = Controls().struct()
    for by_adjoint in (False, True):
        assert eng.tape(ctl, True, 1000, by_adjoint) is None
        assert eng.tape(ctl, False, 0, by_adjoint) is None
        assert eng.tape(ctl, False, (1 << 26) + 1, by_adjoint) is None
        assert eng.tape(Controls(jump=True).struct(), False, 1000, by_adjoint) is None
    assert eng.tape(ctl, False, 1000, False) is None and eng.tape(ctl, False, 1000, True) is not None
    argon = engine(lar_box(), "cuda")
    assert argon.tape(ctl, False, 1000, False) is not None and argon.tape(ctl, False, (1 << 20) + 1, False) is None
