"""The autotuner's remembered choices: one made among other candidates than today's is timed again."""

import json
import types

import pytest

from lumen_amd import autotune
from lumen_amd.api import Controls


@pytest.mark.parametrize("what", ["forward", "adjoint"])
def test_a_choice_among_other_chunks_is_timed_again(tmp_path, monkeypatch, what):
    import torch

    monkeypatch.setenv("LUMEN_AMD_CACHE", str(tmp_path))
    monkeypatch.setattr(torch.cuda, "get_device_name", lambda d: "card")
    run = types.SimpleNamespace(det=types.SimpleNamespace(name="tank"), total=1000, rows=[0] * 3,
                                eng=types.SimpleNamespace(device="cuda"))
    # a file of when the chunks were other ones, and the key did not say which
    (tmp_path / "autotune.json").write_text(json.dumps(
        {f"tank|{what}|photons=1000|sources=3|card": {"chunk": 4096, "blocks_per_cu": 0}}))
    timed = []

    def tune(run, what):
        timed.append(what)
        return Controls(), {(0, 0): 1.0}

    monkeypatch.setattr(autotune, "tune", tune)
    assert autotune.tuned_controls(run, what).chunk == 0 and timed == [what]
    assert autotune.tuned_controls(run, what).chunk == 0 and timed == [what]  # remembered
    monkeypatch.setattr(autotune, "CHUNKS", (0, 64))
    monkeypatch.setattr(autotune, "ADJ_CHUNKS", (0, 64))
    autotune.tuned_controls(run, what)
    assert timed == [what, what]
