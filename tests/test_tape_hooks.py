"""The photon loop's tape and hooks on saved tensors: no hook gets the tape, it is read where the saved tensors come back
as they were, freed with them, and the photons are replayed where they do not."""

import gc
import weakref

import numpy as np
import pytest

import lumen_amd as L
from lumen_amd import autograd
from lumen_amd.detector import example_tank

KEY = "materials/Water/ABSLENGTH"
SRC = L.sources.Point((0.05, 0.0, 0.1), lam=400.0, n_photons=2e5)


def _hooks(torch, name):
    return {"none": lambda: torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t),
            "cpu": torch.autograd.graph.save_on_cpu,
            "half": lambda: torch.autograd.graph.saved_tensors_hooks(lambda t: t.half(), lambda t: t.float())}[name]()


class _Run:
    first_index = first_slot = [0]


@pytest.fixture
def loop(monkeypatch):
    """The photon loop over stand-ins on the CPU: its function, and what they saw."""
    import torch

    seen = {"tapes": []}

    def tape(run, by_adjoint):
        if by_adjoint:
            return None
        t = torch.zeros(1000, dtype=torch.uint8)
        seen["alive"] = weakref.ref(t)
        return t

    def adjoint(run, values, g, tape=None):
        seen["tapes"].append(tape)
        return torch.ones(1, dtype=torch.float64)

    monkeypatch.setattr(autograd, "_tape", tape)
    monkeypatch.setattr(autograd, "_trace", lambda run, values, tape=None: values.double() * 2.0)
    monkeypatch.setattr(autograd, "adjoint", adjoint)
    return autograd._function(), seen


@pytest.mark.parametrize("name,read", [("none", True), ("half", False)])
def test_no_hook_gets_the_tape(loop, name, read):
    import torch

    fn, seen = loop
    packed = []
    x = torch.ones(3, requires_grad=True)
    with _hooks(torch, name):
        with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.dtype) or t, lambda t: t):
            fn.apply(x * 1.0, _Run()).sum()
        y = fn.apply(x * 1.0, _Run())
    assert torch.uint8 not in packed
    y.sum().backward(retain_graph=True)
    y.sum().backward()
    gc.collect()
    assert [t is not None for t in seen["tapes"]] == [read, read]
    seen["tapes"].clear()
    gc.collect()
    assert seen["alive"]() is None  # with the saved tensors, while y lives
    assert y is not None


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["none", "cpu"])
def test_the_gradient_under_hooks(gpu, name):
    import torch

    det = example_tank()

    def grad():
        t = autograd.table_tensor(det.params(), KEY)
        light = autograd.simulate_diff(det, SRC, {KEY: t}, samples=4097, seed=4)
        light.arrivals.sum().backward()
        return t.grad.cpu().numpy()

    alone = grad()
    with _hooks(torch, name):
        under = grad()
    # the same float32 terms added in FP64, a term some ten roundings of 2^-24 where a kernel contracts another product
    assert np.linalg.norm(under - alone) <= 2e-6 * np.linalg.norm(alone)
