"""The packed values' upload is not waited for by the host, and a later call with the same values takes the copy again:
on another stream it is ordered after the copy, whatever stands before that on the first stream."""

import numpy as np
import pytest

import lumen_amd as L
from lumen_amd import api
from lumen_amd.detector import example_tank

SRC = L.sources.Point((0.05, 0.0, 0.1), lam=400.0, n_photons=2e5)
KEY = "materials/Water/ABSLENGTH"


class _Stream:
    def __init__(self):
        self.waited = []

    def wait_event(self, event):
        self.waited.append(event)


class _Event:
    def record(self, stream):
        self.on = stream


class _Copy:
    def __init__(self):
        self.used_on = []

    def record_stream(self, stream):
        self.used_on.append(stream)


def test_another_stream_waits_for_the_copy(monkeypatch):
    import torch

    eng = object.__new__(api.Engine)
    eng.device, eng._uploads = "cuda", {}
    x, y = _Stream(), _Stream()
    now = [x]
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: now[0])
    monkeypatch.setattr(torch.cuda, "Event", _Event)
    monkeypatch.setattr(api, "to_device", lambda a, device: _Copy())
    v = np.arange(5, dtype=np.float32)
    a = eng.upload(v)
    assert eng.upload(v.copy()) is a and not x.waited and not a.used_on  # its own stream: in order already
    now[0] = y
    assert eng.upload(v.copy()) is a
    assert len(y.waited) == 1 and y.waited[0].on is x and a.used_on == [y]
    b = eng.upload(v + 1.0)  # new values, copied on y
    assert b is not a and len(y.waited) == 1
    now[0] = x
    assert eng.upload(v + 1.0) is b and x.waited[-1].on is y and b.used_on == [x]


@pytest.mark.gpu
@pytest.mark.parametrize("first", ["returns", "raises after its upload"])
def test_a_fit_on_a_stream_beside_a_busy_one(gpu, first):
    """A call on a stream that is still busy, then a fit's step on an idle one with the same values and no wait by the
    host: the fit is the fit alone."""
    import torch

    from lumen_amd.autograd import simulate_diff, table_tensor

    det = example_tank()
    n = 4097

    def fit():
        t = table_tensor(det.params(), KEY)
        light = simulate_diff(det, SRC, {KEY: t}, samples=n, seed=4)
        light.arrivals.sum().backward()
        return light.arrivals.detach(), t.grad

    alone = [v.cpu().numpy() for v in fit()]
    eng = api.engine(det)
    x, y = torch.cuda.Stream(), torch.cuda.Stream()
    big = torch.randn((8192, 8192), device="cuda")
    torch.cuda.synchronize()
    eng._uploads.clear()  # the next call copies the values
    with torch.cuda.stream(x):
        for _ in range(20):
            big = big @ big * 1e-3
        if first == "returns":
            L.simulate(det, SRC, samples=n, seed=5)
        else:
            with pytest.raises(ValueError, match="events"):
                L.simulate(det, SRC, samples=n, seed=5, events=0)
    with torch.cuda.stream(y):
        beside = fit()
    torch.cuda.synchronize()
    # FP64 sums of the same terms in another order; the gradient is rounded to float32 once
    np.testing.assert_allclose(beside[0].cpu().numpy(), alone[0], rtol=n * 1.2e-16, atol=0.0)
    np.testing.assert_allclose(beside[1].cpu().numpy(), alone[1], rtol=2.5e-7, atol=0.0)
