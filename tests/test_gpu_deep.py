"""An exit of a volume that lies deep inside its mother skips the test that the mother holds the point past the face
(``deep_in_mother``): the crossings of rays from inside the daughter are those of the same model built without boxes,
which has no such volume, whatever the gap to the mother's face and the mother's form and frame."""

import numpy as np
import pytest

from lumen_amd import _lib
from lumen_amd.api import Engine
from lumen_amd.detector import navarrays, solids
from nav_scenes import rx, rz
from toys import sphere_toy

pytestmark = pytest.mark.gpu

MOTHERS = {"box": solids.box(0.5, 0.4, 0.3), "tube": solids.tube(0.4, 0.3), "orb": solids.orb(0.45),
           "ring": solids.tube(0.6, 0.3, rmin=0.05)}


def _engine(mother, gap, R, monkeypatch, boxes):
    """World / mother (frame R) / a box daughter whose +x face is ``gap`` from the mother's +x extent."""
    m = MOTHERS[mother]
    half = {"box": 0.5, "tube": 0.4, "orb": 0.45, "ring": 0.6}[mother]
    t = np.array([0.1, -0.2, 0.05])
    side = 0.02
    at = np.array([half - gap - side, 0.0, 0.0])
    kinds = [solids.box(2.0, 2.0, 2.0, name="world"), m, solids.box(side, side, side, name="cube")]
    vols = [navarrays.Volume("w", 0, np.eye(3), np.zeros(3), -1, 0), navarrays.Volume("w/m", 1, R, t, 0, 0),
            navarrays.Volume("w/m/c", 2, R, R @ at + t, 1, 0)]
    det = sphere_toy()
    det.nav = navarrays.build(vols, kinds, outside_cls=2)
    det.sensor_of_vol = np.full(4, -1, np.int32)
    if not boxes:
        full = _lib.geometry_struct

        def without(*a):
            g, keep = full(*a)
            g.box_lo = g.box_hi = None
            return g, keep

        monkeypatch.setattr(_lib, "geometry_struct", without)
    return Engine(det, "cuda"), R @ at + t, side


@pytest.mark.parametrize("mother", sorted(MOTHERS))
@pytest.mark.parametrize("gap", [0.0, 1e-6, 3e-5, 3e-4, 1e-2, 0.1])
def test_a_deep_exit_is_the_tested_one(gpu, mother, gap, monkeypatch):
    rng = np.random.default_rng(7)
    R = rz(25.0) @ rx(40.0)
    out = []
    for boxes in (True, False):
        eng, c, side = _engine(mother, gap, R, monkeypatch, boxes)
        rng = np.random.default_rng(7)
        n = 20000
        x = c + (rng.uniform(-1, 1, (n, 3)) * side) @ R.T
        d = rng.normal(size=(n, 3))
        d[: n // 2] = R[:, 0] + 0.2 * d[: n // 2]  # at the near face
        out.append(eng.query(x, d, vol=np.full(n, 2, np.int32)))
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
