"""The range of the pressure (one launch, the last workgroup reduces): rows
shorter, as long and longer than a piece of 2048 cells, more pieces than
workgroups, padding left out, NaN ignored, infinities, all NaN, and repeated
calls.  Minimum and maximum are exact."""
import numpy as np
import pytest

from opensayal_amd import Batch, Fluid
from tests.helpers import make_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H", [(3, 3), (65, 700), (2047, 5), (2048, 511), (2049, 300),
                                 (4100, 1031)])
def test_pressure_range_of_any_field(W, H):
    rng = np.random.default_rng(W)
    with Fluid(make_config(W, H, enable_pressure=1)) as fl, Batch() as bt:
        bt.add(fl)  # a member's range is reduced when it is asked for
        for k in range(4):
            p = rng.uniform(1.0 + k, 5.0, (H, W)).astype(np.float32)  # 0 only in the padding
            if k == 1:
                p = -p
            if k == 2:
                p[rng.random((H, W)) < 0.3] = np.nan
                p[H - 1, W - 1] = np.inf
                p[0, 0] = 2.5
            if k == 3:
                p[:] = np.nan
            fl.set_field("pressure", p)
            want = (np.inf, -np.inf) if k == 3 else (np.nanmin(p), np.nanmax(p))
            assert fl.pressure_range == pytest.approx(want, abs=0.0, rel=0.0)
