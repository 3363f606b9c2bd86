"""The tapes alive take at most their part of a device's free memory: further launches take none, and their adjoint
replays the photons."""

import gc
import types

import numpy as np
import pytest

import lumen_amd as L
from lumen_amd import _lib, api
from lumen_amd.api import Controls
from lumen_amd.detector import example_tank

SRC = L.sources.Point((0.05, 0.0, 0.1), lam=400.0, n_photons=2e5)
KEY = "materials/Water/ABSLENGTH"


class _Sized:
    """The library's lh_tape_size: a byte a photon, written by the forward."""

    def lh_tape_size(self, handle, ctl, has_ref, photons, nbytes, by_adjoint):
        nbytes._obj.value, by_adjoint._obj.value = photons, 0
        return 0


def _engine(device="cpu"):
    eng = object.__new__(api.Engine)
    eng.device, eng.handle = device, None
    return eng


@pytest.fixture
def free(monkeypatch):
    """The device's free memory, the tapes' own less."""
    import torch

    base = sum(h.nbytes for h in api._TAPES)
    size = types.SimpleNamespace(free=0)
    monkeypatch.setattr(api, "FREE_AGE", 0.0)
    monkeypatch.setattr(api, "_FREE", {})
    monkeypatch.setattr(torch.cuda, "mem_get_info",
                        lambda d=None: (size.free + base - sum(h.nbytes for h in api._TAPES), 0))
    return size


def test_tapes_take_their_part(monkeypatch, free):
    import torch

    gc.collect()
    monkeypatch.setattr(_lib, "lib", lambda: _Sized())
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    ctl = Controls().struct()
    a, b = _engine(), _engine()  # two detectors share the device
    n = 1000
    free.free = 3 * n * api.TAPE_PARTS
    got = [e.tape(ctl, False, n, False) for e in (a, b, a, b, a)]
    assert [t is not None for t in got] == [True, True, True, False, False]
    assert all(t.numel() == n for t in got[:3])
    assert a.tape(ctl, False, 1, False) is None
    del got[0]
    gc.collect()
    assert b.tape(ctl, False, n, False) is not None
    free.free = n * api.TAPE_PARTS - 1
    got.clear()
    gc.collect()
    assert a.tape(ctl, False, n, False) is None  # one tape of more than its part


def test_free_memory_is_looked_up_again(monkeypatch, free):
    import torch

    looks = []
    real = torch.cuda.mem_get_info
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda d=None: looks.append(d) or real(d))
    monkeypatch.setattr(_lib, "lib", lambda: _Sized())
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(api, "FREE_AGE", 5.0)
    now = [100.0]
    monkeypatch.setattr(api.time, "monotonic", lambda: now[0])
    gc.collect()
    free.free = 10 * api.TAPE_PARTS
    eng, ctl = _engine(), Controls().struct()
    kept = [eng.tape(ctl, False, 4, False) for _ in range(3)]
    assert [t is not None for t in kept] == [True, True, False] and looks == [0]  # the tapes since are counted
    now[0] += 5.0
    free.free = 12 * api.TAPE_PARTS
    assert eng.tape(ctl, False, 4, False) is not None and looks == [0, 0]


@pytest.mark.gpu
def test_results_kept_for_a_later_backward(gpu, free):
    """Room for two tapes: of five results kept for one backward two hold one, and the gradient is that of five with."""
    import torch

    from lumen_amd.autograd import simulate_diff, table_tensor

    det = example_tank()
    n = 4097

    def grad(room):
        free.free = room
        t = table_tensor(det.params(), KEY)
        lights = [simulate_diff(det, SRC, {KEY: t}, samples=n, seed=s) for s in range(5)]
        held = len(api._TAPES)
        sum(x.arrivals.sum() for x in lights).backward()
        return held, t.grad.cpu().numpy()

    gc.collect()
    free.free = 1 << 40
    size = api.engine(det).tape(Controls().struct(), False, n, False).numel()
    gc.collect()
    kept = len(api._TAPES)
    few, a = grad(2 * size * api.TAPE_PARTS)
    gc.collect()
    assert len(api._TAPES) == kept  # given back by the backward
    all_of_them, b = grad(1 << 40)
    assert (few - kept, all_of_them - kept) == (2, 5)
    # the same float32 terms added in FP64, a term some ten roundings of 2^-24 where a kernel contracts another product
    assert np.linalg.norm(b - a) <= 2e-6 * np.linalg.norm(a)
    torch.cuda.synchronize()
