"""The launch shape a handle starts with follows its grid, sweeps, storage and
pressure: grids on both sides of every change of shape, against the
colour-phase kernel, bit for bit (the same updates in the same order)."""
import numpy as np
import pytest

from tests.helpers import make_config
from tests.test_gpu_parity import pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H,n", [(3, 3, 1), (64, 36, 20), (640, 480, 50), (700, 500, 9),
                                   (1001, 563, 13), (1280, 720, 12), (1921, 1085, 7),
                                   (2049, 1150, 8), (2560, 1440, 11)])
@pytest.mark.parametrize("storage,pressure", [(0, 0), (0, 1), (2, 0), (1, 1)])
def test_starting_shape_matches_colour_phases(W, H, n, storage, pressure):
    cfg = make_config(W, H, projection_n=n, storage=storage, enable_pressure=pressure,
                      obstacle_radius=min(W, H) / 8.0)
    out = []
    for colour in (False, True):
        fl, _ = pair(cfg, seed=41)
        if colour:
            fl.set_tuning(projection_kernel=0)
        else:
            assert fl.projection_kernel == 2
        fl.project()
        out.append([fl.get_field(f) for f in ("vel_x", "vel_y", "pressure")[:2 + pressure]])
    for a, b in zip(*out):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
