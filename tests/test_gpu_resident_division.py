"""Resident projections whose pressure sums divide by d_t (0, or 2 and more in
magnitude: no double reciprocal) against the oracle, bit for bit: both region
heights the kernel has, several tiles each way, every storage type, a short
last stage and launches one after the other."""
import numpy as np
import pytest

from tests.helpers import make_config
from tests.test_gpu_parity import pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", [0, 1, 2])
@pytest.mark.parametrize("rows,k", [(4, 2), (8, 5)])
@pytest.mark.parametrize("d_t,kw", [(2.0, {}), (-3.7, dict(density=0.7, enable_drain=0)),
                                    (2.5, dict(cell_size=2.0)), (0.0, {})])
def test_dividing_resident_equals_oracle(storage, rows, k, d_t, kw):
    cfg = make_config(250, 230, projection_n=13, enable_pressure=1, d_t=d_t, storage=storage,
                      wind_speed=0.01, g=-0.01, obstacle_center_x=100, obstacle_center_y=104,
                      obstacle_radius=20.5, **kw)
    fl, o = pair(cfg, seed=21)
    fl.set_tuning(projection_kernel=3, tile_width=128 - 4 * k, tile_height=8 * rows - 4 * k,
                  sweeps_per_launch=k)
    assert fl.projection_kernel == 3 and fl.launches_per_call(13) == 1
    if storage == 0:  # (alone it takes the state as set, which is not rounded in the oracle)
        fl.project()
        o.projection()
    fl.step(3)
    o.update(steps=3)
    for name, attr in (("vel_x", "u"), ("vel_y", "v"), ("smoke", "smoke"), ("pressure", "p")):
        got, ref = fl.get_field(name), getattr(o, attr)
        assert np.array_equal(np.isnan(got), np.isnan(ref)), name
        ok = ~np.isnan(ref)
        assert np.array_equal(got[ok].view(np.uint32), ref[ok].view(np.uint32)), name
