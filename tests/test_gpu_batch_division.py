"""Batch members whose pressure sums divide by d_t (0, or 2 and more in
magnitude: no double reciprocal) step in the persistent launch: the bits of
the same handle alone and of the oracle, beside members that take the
reciprocal, in every storage type and register shape."""
import numpy as np
import pytest

from opensayal_amd import Batch
from oracle.oracle import OracleFluid
from tests.helpers import make_config
from tests.test_gpu_batch import assert_same, started, state
from opensayal_amd import workloads as wl

pytestmark = pytest.mark.gpu


def config(W, H, n, d_t, storage, **kw):
    return make_config(W, H, projection_n=n, enable_pressure=1, d_t=d_t, storage=storage,
                       wind_speed=0.01, g=-0.01, obstacle_center_x=W // 3,
                       obstacle_center_y=H // 2, obstacle_radius=6.5, **kw)


@pytest.mark.parametrize("storage", [0, 1, 2])
@pytest.mark.parametrize("rows,k,occ", [(12, 10, 2), (8, 5, 1), (8, 6, 2)])
def test_dividing_members_equal_alone_and_oracle(storage, rows, k, occ):
    cfgs = [config(77, 53, 13, 2.0, storage), config(150, 110, 20, 0.05, storage),
            config(131, 60, 11, -3.7, storage, density=0.7), config(64, 36, 7, 0.0, storage),
            config(140, 100, 12, 2.5, storage, cell_size=2.0, enable_drain=0)]
    batched = [started(c, 40 + i) for i, c in enumerate(cfgs)]
    alone = [started(c, 40 + i) for i, c in enumerate(cfgs)]
    with Batch() as b:
        b.set_tuning(rows=rows, sweeps_per_tile=k, occupancy=occ)
        for fl in batched:
            b.add(fl)
        b.step(3)
        for i, (x, y) in enumerate(zip(batched, alone)):
            y.step(3)
            assert_same(state(x), state(y), f"sim {i} d_t={cfgs[i].d_t}")
            o = OracleFluid(cfgs[i])
            u, v, s = wl.initial_state(cfgs[i], 40 + i)
            o.set_state(u=u, v=v, smoke=s)
            o.update(steps=3)
            for name, attr in (("vel_x", "u"), ("vel_y", "v"), ("smoke", "smoke"),
                               ("pressure", "p")):
                got, ref = x.get_field(name), getattr(o, attr)
                assert np.array_equal(np.isnan(got), np.isnan(ref)), name
                ok = ~np.isnan(ref)
                assert np.array_equal(got[ok].view(np.uint32), ref[ok].view(np.uint32)), name
