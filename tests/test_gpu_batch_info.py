"""What a Fluid says of itself after a batch has changed it: a resident shape whose
halo exchange the budget has no room for, and the shape that the batch's
autotuner picks for a member on its own graphs."""
import ctypes

import pytest

from opensayal_amd import Batch, Fluid, device_bytes
from opensayal_amd._abi import OsyFluidInfo, check, lib
from tests.helpers import make_config

pytestmark = pytest.mark.gpu


def of_library(fl):
    info = OsyFluidInfo()
    check(lib().osy_fluid_get_info(fl._h, ctypes.byref(info)))
    return info.projection_kernel, info.sweeps_per_launch, info.device_bytes


def of_object(fl):
    return fl.projection_kernel, fl.sweeps_per_launch, fl.device_bytes


def test_info_follows_the_batch():
    cfg = make_config(250, 230, projection_n=20)
    for budget in (device_bytes(cfg), 0):
        with Fluid(cfg) as fl, Batch(budget) as b:
            fl.set_tuning(projection_kernel=3, tile_width=116, tile_height=52,
                          sweeps_per_launch=3)
            b.set_per_grid_cells(1)
            b.add(fl)
            assert of_object(fl) == of_library(fl)
            assert (fl.projection_kernel, fl.device_bytes == device_bytes(cfg)) == (
                (2, True) if budget else (3, False))
            b.autotune()
            assert of_object(fl) == of_library(fl)


def test_closed_member_does_not_matter():
    cfg = make_config(64, 36, projection_n=5)
    with Fluid(cfg) as fl, Batch() as b:
        gone = Fluid(cfg)
        b.add(fl)
        b.add(gone)
        gone.close()
        b.autotune()
        b.step(2)
