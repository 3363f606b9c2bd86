"""Host arrays are not uploaded inside a graph's capture: the copy comes from pinned memory that is handed out again after
the call, so a replay would read another array's bytes."""

import numpy as np
import pytest

import lumen_amd as L
from lumen_amd import api, readout
from lumen_amd.detector import example_tank

SRC = L.sources.Point((0.05, 0.0, 0.1), lam=400.0, n_photons=2e5)


def test_no_upload_while_capturing(monkeypatch):
    import torch

    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    with pytest.raises(RuntimeError, match="graph is captured"):
        api.to_device(np.zeros(3), "cuda")
    np.testing.assert_array_equal(api.to_device(np.arange(3), "cpu").numpy(), np.arange(3))


@pytest.mark.gpu
def test_a_captured_readout_is_refused(gpu):
    import torch

    det = example_tank()
    light = L.simulate(det, SRC, samples=4097, seed=4)
    pe = readout.pe(light, det.params(), det).cpu().numpy()
    torch.cuda.synchronize()
    with pytest.raises(RuntimeError, match="graph is captured"):
        with torch.cuda.graph(torch.cuda.CUDAGraph()):
            torch.zeros(1, device="cuda").add_(1.0)  # the capture holds something beside the refused call
            readout.pe(light, det.params(), det)
    np.testing.assert_array_equal(readout.pe(light, det.params(), det).cpu().numpy(), pe)
