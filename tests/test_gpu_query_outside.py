"""``Engine.query`` of rays in a given volume that does not hold their start: they leave it at once, into whatever holds
the start, also where the volume lies deep inside its mother (``deep_in_mother``) and the start outside of both."""

import numpy as np
import pytest

from nav_scenes import rx, rz
from test_gpu_deep import MOTHERS, _engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mother", sorted(MOTHERS))
def test_a_start_outside_its_volume(gpu, mother, monkeypatch):
    out = []
    for boxes in (True, False):  # without boxes no volume is deep: every exit's mother is tested
        eng, c, side = _engine(mother, 0.1, rz(25.0) @ rx(40.0), monkeypatch, boxes)
        rng = np.random.default_rng(8)
        n = 20000
        x = rng.uniform(-1.5, 1.5, (n, 3))
        x[: n // 4] = c + rng.uniform(-2.0, 2.0, (n // 4, 3)) * side  # about the volume itself
        out.append(eng.query(x, rng.normal(size=(n, 3)), vol=np.full(n, 2, np.int32)))
    outside = out[0][4] == 0
    assert outside.mean() > 0.3  # in the world, outside the mother
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
